"""The mid-M weight-quant kernel (nz_mid) on the GPU: int4 / int8 NZ and int8 [N, K] weights, and row-major weights
cast to NZ for it, with every K split forced that the debug plan offers.

Row counts at the edges of its row tiles (16-row pieces, 96-row tiles, 64 with half-step groups), an N of a partial
256-column tile and one of a single 16-column block, K of one step and of uneven splits, groups of one step, several
steps, half a step and all of K.  Held to the op's rtol = atol = 1e-2 bar against the float64 oracle; scales differ
per group and channel and rows of x past M are NaN.
"""
import ctypes

import pytest
import torch

from op_plugin_amd import workloads as W

pytestmark = pytest.mark.gpu
CODE = {torch.float16: 1, torch.bfloat16: 2}
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import op_plugin_amd
    yield op_plugin_amd
    op_plugin_amd.debug_set_plan("")


def _inputs(int4, M, N, K, group, offset, dtype, bias, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.full((M + 5, K), float("nan"), dtype=dtype)
    x[:M] = torch.randn((M, K), generator=g).to(dtype)
    w = torch.randint(*((-8, 8) if int4 else (-127, 128)), (K, N), generator=g, dtype=torch.int8)
    rows = (K // group, N) if group else (N,)
    scale = ((2e-2 if int4 else 1.2e-3) * (0.25 + 0.75 * torch.rand(rows, generator=g))).half()
    off = (2 * torch.rand(rows, generator=g) - 1).half() if offset else None
    b = torch.randn(N, generator=g).to(dtype) if bias else None
    return x, w, scale, off, b


def _ref(oracle, int4, x, w, scale, off, b, group, dtype):
    return W.from_bits(oracle.weight_quant_bmm(
        W.bits(x), CODE[dtype], (W.int4_pack_cpu(w) if int4 else w).numpy(), W.bits(scale),
        None if off is None else W.bits(off), 1, group, bias=None if b is None else W.bits(b), bias_dtype=CODE[dtype],
        out_dtype=CODE[dtype]), dtype).float()


def _weight(ops, w, int4, layout):
    if layout == "nk":
        return w.t().contiguous().to(DEV).t()
    wd = ops.npu_convert_weight_to_int4pack(w.to(DEV)) if int4 else w.to(DEV)
    return ops.npu_format_cast(wd, ops.ACL_FORMAT_FRACTAL_NZ) if layout == "nz" else wd


CASES = [
    # int4, layout, M, N, K, group, offset, dtype, bias
    (True, "nz", 17, 16, 128, 128, True, torch.bfloat16, False),     # one step, one 16-column block
    (True, "nz", 33, 272, 640, 128, True, torch.float16, True),      # three row pieces, a 16-column tail
    (True, "nz", 65, 256, 1408, 128, False, torch.bfloat16, False),  # five row pieces, 11 steps
    (True, "nz", 96, 528, 896, 0, True, torch.float16, False),       # a whole 96-row tile, one group over K
    (True, "nz", 97, 512, 1024, 256, True, torch.bfloat16, True),    # two row tiles, two-step groups
    (True, "nz", 200, 304, 768, 64, True, torch.bfloat16, False),    # half-step groups, four 64-row tiles
    (True, "nz", 64, 48, 2176, 64, False, torch.float16, True),
    (False, "nz", 20, 80, 64, 0, True, torch.bfloat16, False),       # one 64-row step
    (False, "nz", 100, 272, 64 * 13, 64, True, torch.float16, True),
    (False, "nz", 130, 256, 64 * 20, 128, False, torch.bfloat16, False),
    (False, "nk", 50, 272, 128 * 7, 128, True, torch.bfloat16, True),
    (False, "nk", 300, 64, 128 * 5, 0, False, torch.float16, False),
    (True, "kn", 70, 272, 1408, 128, True, torch.bfloat16, False),   # cast to NZ first
    (False, "kn", 70, 272, 64 * 13, 0, True, torch.float16, True),
]


@pytest.mark.parametrize("int4,layout,M,N,K,group,offset,dtype,bias", CASES)
def test_nz_mid(ops, oracle, int4, layout, M, N, K, group, offset, dtype, bias):
    print(f"[case] int4={int4} {layout} M={M} N={N} K={K} G={group} offset={offset} {dtype} bias={bias}", flush=True)
    x, w, scale, off, b = _inputs(int4, M, N, K, group, offset, dtype, bias, seed=M + K)
    ref = _ref(oracle, int4, x[:M], w, scale, off, b, group, dtype)
    wd = _weight(ops, w, int4, layout)
    steps = K // (128 if int4 else 64)
    dev = lambda t: None if t is None else t.to(DEV)
    for split in sorted({1, 2, 3, min(7, steps), min(16, steps)}):
        if split > steps:
            continue
        ops.debug_set_plan(f"nz_mid={split}")
        out = ops.npu_weight_quant_batchmatmul(x.to(DEV)[:M], wd, dev(scale), dev(off), bias=dev(b),
                                               antiquant_group_size=group)
        torch.testing.assert_close(out.cpu().float(), ref, rtol=1e-2, atol=1e-2, msg=lambda m: f"split {split}: {m}")
    ops.debug_set_plan("")


def test_nz_mid_workspace_and_capture(ops):
    """The planned shape reports its partials, runs on a workspace of any contents, and replays in a graph."""
    M, N, K, G = 100, 4096, 4096, 128
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn((M, K), generator=g, device=DEV).bfloat16()
    w = torch.randint(-8, 8, (K, N), generator=g, device=DEV, dtype=torch.int8)
    nz = ops.npu_format_cast(ops.npu_convert_weight_to_int4pack(w), ops.ACL_FORMAT_FRACTAL_NZ)
    s = (0.005 + 0.015 * torch.rand((K // G, N), generator=g, device=DEV)).half()
    ref = ops.npu_weight_quant_batchmatmul(x, nz, s, antiquant_group_size=G)
    L, n = ops.abi(), ctypes.c_size_t(0)
    assert L.qk_weight_quant_bmm_workspace_size(M, N, K, ops.QK_I4_NZ, G, ctypes.byref(n)) == 0
    assert n.value > 4096 + M * N * 4  # at least two splits' partials
    for fill in (0, 0xFF):
        ws = torch.full((n.value,), fill, dtype=torch.uint8, device=DEV)
        out = torch.empty_like(ref)
        rc = L.qk_weight_quant_bmm(x.data_ptr(), ops.QK_BF16, nz.data_ptr(), ops.QK_I4_NZ, s.data_ptr(), None, ops.QK_F16,
                                   M, N, K, G, None, 0, out.data_ptr(), ops.QK_BF16, ws.data_ptr(), n.value,
                                   torch.cuda.current_stream().cuda_stream)
        assert rc == 0, ops.last_error()
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.npu_weight_quant_batchmatmul(x, nz, s, antiquant_group_size=G)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16))
        eager = ops.npu_weight_quant_batchmatmul(x, nz, s, antiquant_group_size=G)
        assert torch.equal(eager.view(torch.int16), ref.view(torch.int16))


def test_long_group_sums(ops, oracle):
    """Prefill with one group over K: the wave-per-row sums of x, rows no multiple of the workgroup's."""
    for M, K in ((1027, 2048), (1027, 512 + 128)):
        x, w, scale, off, _ = _inputs(True, M, 4096, K, 0, True, torch.bfloat16, False, seed=K)
        wd = _weight(ops, w, True, "nz")
        ops.debug_set_plan("nz_mid=0")
        out = ops.npu_weight_quant_batchmatmul(x.to(DEV)[:M], wd, scale.to(DEV), off.to(DEV))
        ops.debug_set_plan("")
        rows = torch.tensor([0, 1, 511, M - 2, M - 1])
        ref = _ref(oracle, True, x[rows], w, scale, off, None, 0, torch.bfloat16)
        torch.testing.assert_close(out.cpu()[rows].float(), ref, rtol=1e-2, atol=1e-2)
