"""Weight-quant decode on K that no even split covers, on the GPU.

* NZ / [N, K] weights (w4nz_decode's ragged form): K of an uneven number of 128-row superblocks per wave, one
  superblock, more than 16 waves of 8, an int8 K that ends in half a superblock, 64-row groups; row counts at the
  edges of its x slots (4 / 5) and row blocks (16 / 17, 64).
* Row-major weights (w4_stream): a last K split that reaches past K, whole 32-row blocks short.

Every output is held to the op's rtol = atol = 1e-2 bar against the float64 oracle.  Scales differ per group and
channel, and rows of x beyond the call's are NaN, so a superblock, group or row taken twice, left out or read from
the wrong place shows.
"""
import numpy as np
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
    return op_plugin_amd


def _case(ops, oracle, int4, layout, M, N, K, group, offset, dtype, seed):
    print(f"[case] int4={int4} {layout} M={M} N={N} K={K} G={group} offset={offset} {dtype}", flush=True)
    g = torch.Generator().manual_seed(seed)
    xfull = torch.full((M + 3, K), float("nan"), dtype=dtype)  # rows past M hold NaN
    xfull[:M] = torch.randn((M, K), generator=g).to(dtype)
    lo, hi = (-8, 8) if int4 else (-127, 128)
    w = torch.randint(lo, hi, (K, N), generator=g, dtype=torch.int8)
    rows = (K // group, N) if group else (N,)
    top = 2e-2 if int4 else 1.2e-3
    scale = (top * (0.25 + 0.75 * torch.rand(rows, generator=g))).half()
    off = (2 * torch.rand(rows, generator=g) - 1).half() if offset else None
    if int4:
        wd = ops.npu_convert_weight_to_int4pack(w.to(DEV))
        wref = W.int4_pack_cpu(w).numpy()
    else:
        wd = w.t().contiguous().to(DEV).t() if layout == "nk" else w.to(DEV)
        wref = w.numpy()
    if layout == "nz":
        wd = ops.npu_format_cast(wd, ops.ACL_FORMAT_FRACTAL_NZ)
    out = ops.npu_weight_quant_batchmatmul(xfull.to(DEV)[:M], wd, scale.to(DEV), None if off is None else off.to(DEV),
                                           antiquant_group_size=group)
    ref = oracle.weight_quant_bmm(W.bits(xfull[:M]), CODE[dtype], wref, W.bits(scale),
                                  None if off is None else W.bits(off), 1, group, out_dtype=CODE[dtype])
    torch.testing.assert_close(out.cpu().float(), W.from_bits(ref, dtype).float(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("int4,layout,M,N,K,group,offset,dtype", [
    (True, "nz", 1, 48, 128 * 17, 128, True, torch.bfloat16),     # two superblocks per wave, the last wave one
    (True, "nz", 4, 80, 128 * 43, 128, False, torch.float16),     # three per wave, four in flight
    (True, "nz", 5, 16, 128 * 43, 0, True, torch.bfloat16),       # sixteen-row slots, one group over K
    (True, "nz", 3, 32, 128 * 131, 128, True, torch.bfloat16),    # more than 16 waves of 8
    (True, "nz", 16, 32, 128 * 131, 128 * 131, False, torch.float16),
    (True, "nz", 17, 64, 128 * 86, 256, True, torch.bfloat16),    # a second row block of one row
    (True, "nz", 64, 48, 128 * 19, 128, True, torch.float16),
    (True, "nz", 2, 16 * 1025, 128 * 5, 64, True, torch.bfloat16),  # 64-row groups, four and five blocks per workgroup
    (True, "nz", 9, 64, 128 * 33, 64, False, torch.float16),
    (True, "nz", 1, 32, 128, 64, True, torch.bfloat16),           # one superblock of two groups
    (False, "nz", 1, 48, 64 * 65, 0, True, torch.bfloat16),       # ends in half a superblock
    (False, "nz", 6, 16 * 513, 64 * 7, 64, True, torch.float16),  # half a superblock, three blocks per workgroup
    (False, "nz", 16, 32, 64, 0, False, torch.bfloat16),          # half a superblock alone
    (False, "nz", 33, 32, 128 * 43, 128, True, torch.bfloat16),
    (False, "nk", 3, 64, 128 * 33, 128, True, torch.bfloat16),
    (False, "nk", 16, 48, 128 * 107, 0, False, torch.float16),
    (False, "nk", 70, 32, 128 * 35, 128, True, torch.bfloat16),   # two row chunks
    (False, "nk", 3, 64, 64 * 65, 64, True, torch.bfloat16),      # transposed: the row-major stream's ragged K
])
def test_nz_decode_ragged(ops, oracle, int4, layout, M, N, K, group, offset, dtype):
    _case(ops, oracle, int4, layout, M, N, K, group, offset, dtype, seed=K + M)


@pytest.mark.parametrize("int4,M,N,K,group,offset,dtype", [
    (True, 1, 264, 128 * 9, 128, True, torch.bfloat16),      # half-line strips, the last split one wave long
    (True, 16, 272, 128 * 43, 128, False, torch.float16),    # whole-line strips
    (True, 7, 256, 128 * 86, 256, True, torch.bfloat16),
    (True, 16, 64, 4160, 0, True, torch.bfloat16),           # one group, K half a wave's range short
    (True, 3, 136, 4160, 64, False, torch.float16),          # 64-row groups, half a wave's range
    (True, 16, 64, 32 * 33, 32, True, torch.bfloat16),       # 32-row groups, one block past a whole split
    (True, 2, 40, 32, 0, True, torch.bfloat16),              # one 32-row block in all
    (False, 1, 48, 128 * 43, 128, True, torch.bfloat16),     # whole rows per wave
    (False, 16, 24, 4160, 0, False, torch.float16),          # half rows per wave
    (False, 5, 100, 128 * 11, 128, True, torch.bfloat16),    # quarter rows
    (False, 20, 48, 4160, 64, True, torch.bfloat16),         # slices of 16 rows
])
def test_row_major_stream_ragged(ops, oracle, int4, M, N, K, group, offset, dtype):
    _case(ops, oracle, int4, "kn", M, N, K, group, offset, dtype, seed=K + M)


def test_row_major_stream_ragged_abi_scratch(ops):
    """The no-allocation entry point takes the ragged splits on its own scratch and gives the op's bits."""
    M, N, K = 16, 4096, 11008
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn((M, K), generator=g, device=DEV).bfloat16()
    w4 = ops.npu_convert_weight_to_int4pack(torch.randint(-8, 8, (K, N), generator=g, device=DEV, dtype=torch.int8))
    s = (0.02 * torch.rand((K // 128, N), generator=g, device=DEV) + 0.005).half()
    ref = ops.npu_weight_quant_batchmatmul(x, w4, s, antiquant_group_size=128)
    out = torch.empty_like(ref)
    rc = ops.abi().qk_weight_quant_bmm_noalloc(x.data_ptr(), ops.QK_BF16, w4.data_ptr(), ops.QK_I32, s.data_ptr(),
                                               None, ops.QK_F16, M, N, K, 128, None, 0, out.data_ptr(), ops.QK_BF16,
                                               torch.cuda.current_stream().cuda_stream)
    assert rc == 0, ops.last_error()
    assert np.array_equal(W.bits(out.cpu()), W.bits(ref.cpu()))
