"""W8A8 on shapes with a ragged N or K, bit for bit on the GPU.

The direct-to-LDS prefill kernel (whole tiles, K splits on 256- and 128-row tiles), the mid-M kernel and the decode
split stream on an N that is no multiple of their column tiles and a K that is no multiple of their stages, rings or
splits: the last column tile, the K tail and the short last split.  int32 outputs are held to the exact accumulator
(float64 products on the CPU: every sum is below 2^53), bf16 / fp16 / int8 outputs to the oracle's epilogue of it.
The rows of x1 past M hold 127 and the weight sits inside a larger buffer of 127s, so a read past an edge that is
used shows.
"""
import numpy as np
import pytest
import torch

from op_plugin_amd import workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import op_plugin_amd
    return op_plugin_amd


SHAPES = [
    # M, N, K: qmm_mid (M <= 256)
    (33, 128, 320),      # one stage and a quarter
    (64, 64, 16),        # a K tail alone
    (20, 192, 4160),     # decode rows; K of no 128-row stages
    (200, 128, 1408),    # K of half stages, several row blocks
    # decode split stream on [K,N]
    (5, 256, 128 * 43),
    (16, 512, 128 * 107),
    (32, 256, 128 * 11),
    # 128-row K splits past 32 rows, 256- and 128-row splits past 256 rows, whole tiles
    (100, 272, 13696),
    (128, 528, 11008),
    (300, 256, 11008),
    (300, 1296, 4160),
    (513, 1040, 1376),
    (129, 8272, 2064),
    (700, 272, 5504),
    (257, 49184, 320),   # 2 x 193 whole tiles: no split
    (300, 1536, 5120),   # eight even K ranges of no whole rings: seven run
    (512, 1536, 5120),
]


# [K,N] rows of 8-byte alignment on the split stream: every row tile, one and two blocks of columns, a last piece of
# 8 columns, splits of one and several lengths; 8 columns alone; without a split (129 column tiles); and the tiled
# kernel's side of the rule
HALF_SHAPES = [
    (1, 1000, 4096),
    (16, 264, 1408),
    (17, 520, 1024),
    (33, 8, 640),
    (64, 1000, 13696),
    (128, 248, 5504),
    (100, 1000, 4096),
    (3, 32776, 2048),
    (16, 1000, 512),
    (17, 1000, 512),
]


@pytest.mark.parametrize("M,N,K", HALF_SHAPES)
def test_w8a8_8_byte_rows(ops, oracle, M, N, K):
    test_w8a8_ragged(ops, oracle, "kn", M, N, K)


@pytest.mark.parametrize("layout", ["kn", "nk", "nz"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_w8a8_ragged(ops, oracle, layout, M, N, K):
    if layout == "nz" and K % 64:
        pytest.skip("the NZ cast takes whole 64-row blocks")
    print(f"[case] {layout} M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    xfull = torch.full((M + 2, K), 127, dtype=torch.int8)
    xfull[:M] = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8)
    x = xfull[:M]
    w = torch.randint(-128, 128, (K, N), generator=g, dtype=torch.int8)
    acc = (x.double() @ w.double()).to(torch.int64).to(torch.int32)
    if layout == "nz":
        wd = ops.npu_format_cast(w.to(DEV), ops.ACL_FORMAT_FRACTAL_NZ)
    else:
        src = w.t() if layout == "nk" else w
        buf = torch.full((src.numel() + 4096,), 127, dtype=torch.int8)
        buf[: src.numel()] = src.reshape(-1)
        wd = buf.to(DEV)[: src.numel()].reshape(src.shape)
        wd = wd.t() if layout == "nk" else wd
    xd = xfull.to(DEV)[:M]
    scale = (1e-3 + 9e-3 * torch.rand(N, generator=g))
    pt = 0.01 + 0.02 * torch.rand(M, generator=g)
    bias = (0.1 * torch.randn(N, generator=g)).to(torch.bfloat16)
    offset = torch.rand(N, generator=g) * 8 - 4
    ibias = torch.randint(-1000, 1000, (N,), generator=g, dtype=torch.int32)
    a = acc.numpy()

    out = ops.npu_quant_matmul(xd, wd, scale.to(DEV), output_dtype=torch.int32)
    assert np.array_equal(out.cpu().numpy(), a)
    for dt, code in ((torch.bfloat16, oracle.BF16), (torch.float16, oracle.F16)):
        out = ops.npu_quant_matmul(xd, wd, scale.to(DEV), pertoken_scale=pt.to(DEV), bias=bias.to(DEV), output_dtype=dt)
        ref = oracle.quant_matmul_epilogue(a, scale.numpy(), pertoken=pt.numpy(), bias=W.bits(bias),
                                           bias_dtype=oracle.BF16, out_dtype=code)
        assert np.array_equal(W.bits(out.cpu()), ref)
    out = ops.npu_quant_matmul(xd, wd, (scale * 1e-2).to(DEV), offset=offset.to(DEV), bias=ibias.to(DEV),
                               output_dtype=torch.int8)
    ref = oracle.quant_matmul_epilogue(a, (scale * 1e-2).numpy(), offset=offset.numpy(), bias=ibias.numpy(),
                                       bias_dtype=oracle.I32, out_dtype=oracle.I8)
    assert np.array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize("M,N,K", [(40, 1000, 4096), (300, 1000, 512 * 5), (1100, 72, 2064), (3, 8, 48)])
def test_w8a8_nk_columns_of_eight(ops, M, N, K):
    """[N,K] rows: any N of whole 8-column stores."""
    print(f"[case] nk M={M} N={N} K={K}", flush=True)
    g = torch.Generator().manual_seed(N)
    x = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8)
    out = ops.npu_quant_matmul(x.to(DEV), w.to(DEV).t(), torch.ones(1, device=DEV), output_dtype=torch.int32)
    assert np.array_equal(out.cpu().numpy(), (x.double() @ w.t().double()).numpy().astype(np.int32))
    pt = (1e-3 * (1 + torch.rand(M, generator=g))).to(DEV)
    h = ops.npu_quant_matmul(x.to(DEV), w.to(DEV).t(), torch.ones(1, device=DEV), pertoken_scale=pt,
                             output_dtype=torch.bfloat16)
    assert torch.equal(h, (out.float() * pt[:, None]).to(torch.bfloat16))


@pytest.mark.parametrize("M", [2, 40])
def test_w8a8_8_byte_column_view(ops, M):
    """[K,N]: columns 8.. of a wider tensor; rows 16-byte strides apart that start at 8-byte alignment."""
    g = torch.Generator().manual_seed(M)
    x = torch.randint(-128, 128, (M, 2048), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (2048, 288), generator=g, dtype=torch.int8)
    out = ops.npu_quant_matmul(x.to(DEV), w.to(DEV)[:, 8:280], torch.ones(1, device=DEV), output_dtype=torch.int32)
    assert np.array_equal(out.cpu().numpy(), (x.double() @ w[:, 8:280].double()).numpy().astype(np.int32))
