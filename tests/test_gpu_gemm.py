"""GPU parity of the projection GEMM (gdn_gemm_bf16): C = A B^T with bf16
operands and fp32 accumulation against an fp32 CPU matmul of the same bf16
values, on the GDN layer's projection shapes (in_proj over the concatenated
qkv / z / b / a weights, out_proj) and ragged edges; the fused gate epilogue
against fused_g_beta on the b / a columns."""
import math

import pytest
import torch

from helpers import BF16, bf16_step

pytestmark = pytest.mark.gpu


def _check(c, ref, scale, tag):
    """Each element within one bf16 step of the fp32 reference plus the fp32
    summation-order slack 2^-16 (|A| |B|^T) (the reference and the kernel add
    the K products in different orders; near-zero results carry that absolute
    error), and elements that are not the rounded reference rare."""
    c, ref = c.float().cpu(), ref.float()
    d = (c - ref).abs()
    bound = bf16_step(ref) + scale * 2.0 ** -16
    assert bool((d <= bound).all()), f"{tag}: max |diff| / bound {float((d / bound).max()):.2f}"
    flips = (c != ref.to(BF16).float()).float().mean().item()
    assert flips < 2e-2, f"{tag}: {flips:.2e} of elements are not the rounded reference"


def _ref(a, w):
    return a.float() @ w.float().t(), a.float().abs() @ w.float().abs().t()


# 64 x 64 tiles: (256, 256), (300, 200); with the deeper load pipeline (K >= 1024):
# (1, 8224); 64 x 128: (1000, 2080), (4111, 333); deeper: (300, 8224, 1024) (16
# steps, ragged rows).  The ring kernel: (17, 2048), (256, 2048) (the decode
# out_proj), (100, 2000, 1088) (17 steps dealt to four waves).  The 8-wave kernel:
# (256, 8224) (the decode in_proj, as 130 blocks of 128 x 128), (17000, 2048) (512
# whole tiles and 24 as quarters), (8190, 2047) (one exact round), (17000, 8224)
# (2211 whole tiles).
@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (300, 200, 128), (1, 8224, 2048), (17, 2048, 2048), (256, 2048, 2048),
                                   (100, 2000, 1088), (1000, 2080, 512), (4111, 333, 192), (256, 8224, 2048),
                                   (300, 8224, 1024), (17000, 2048, 256), (8190, 2047, 128), (17000, 8224, 128)])
def test_gemm_against_fp32_matmul(pkg, dev, M, N, K):
    gen = torch.Generator().manual_seed(M * 7 + N)
    a = torch.randn(M, K, generator=gen).to(BF16)
    w = (torch.randn(N, K, generator=gen) / math.sqrt(K)).to(BF16)
    ref, sc = _ref(a, w)
    c = pkg.ops.linear(a.to(dev), w.to(dev))
    _check(c, ref, sc, f"gemm {M}x{N}x{K}")


# 64 x 128 tiles of a short K with ragged rows and columns (the first three); whole
# tiles of the 8-wave kernel with a tail of quarters, an empty one past M, and of an
# uneven round; its K restriction (192: gemm_tn_kernel at 256 and 192 rows); the
# ring kernel at 16 and 32 rows, and 64 x 64 tiles, with 16, 17 and 33 steps (dealt
# to four waves: uneven).  Hv > 0: the columns go to four parts with gate outputs
# (b and a the last 2 Hv columns).
@pytest.mark.parametrize("M,N,K,Hv", [(1949, 2048, 128, 0), (1100, 4000, 256, 16), (1153, 2072, 384, 4),
                                      (4100, 4008, 384, 4), (4500, 3000, 256, 0), (8190, 2047, 192, 0),
                                      (17000, 2048, 192, 0), (1, 2048, 1024, 0), (16, 2056, 1088, 4),
                                      (37, 2048, 2112, 16), (100, 2000, 1024, 8), (200, 2056, 1088, 4),
                                      (250, 1000, 2112, 4)])
def test_gemm_kernel_edges(pkg, dev, M, N, K, Hv):
    gen = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K, generator=gen).to(BF16)
    w = (torch.randn(N, K, generator=gen) / math.sqrt(K)).to(BF16)
    if not Hv:
        c = pkg.ops.linear(a.to(dev), w.to(dev))
        _check(c, *_ref(a, w), f"gemm {M}x{N}x{K}")
        return
    A_log = (torch.rand(Hv, generator=gen) * math.log(16)).to(dev)
    dt_bias = (torch.rand(Hv, generator=gen) * 2 - 1).to(dev)
    first = (N - 2 * Hv) // 32 * 16
    widths = [first, N - 2 * Hv - first, Hv, Hv] if Hv % 16 == 0 else [first, 32, N - first - 32]
    parts, g, beta = pkg.ops.linear_cols(a.to(dev), w.to(dev), widths,
                                         gates={"gate_col": N - 2 * Hv, "A_log": A_log, "dt_bias": dt_bias})
    c = torch.cat(parts, 1)
    _check(c, *_ref(a, w), f"gemm parts {M}x{N}x{K}")
    g2, beta2 = pkg.ops.fused_g_beta(c[:, N - 2 * Hv:N - Hv].contiguous(), c[:, N - Hv:].contiguous(), A_log, dt_bias,
                                     None)
    torch.cuda.synchronize()
    assert torch.equal(g, g2) and torch.equal(beta.view(torch.int16), beta2.view(torch.int16))


# The 8-wave kernel without whole tiles, over the 128 x 128 blocks of C: 3 x 65
# blocks with ragged edges, 16 x 16, 9 x 28 and 10 x 17 (a partial last group of
# rows), 1 x 256 with K of 2 steps; K of 14, 20 and 22 steps (a last round of four
# steps that ends after two).  Hv > 0: four parts with gate outputs.
@pytest.mark.parametrize("M,N,K,Hv", [(300, 8224, 1280, 16), (1949, 2048, 896, 0), (1100, 3500, 896, 4),
                                      (1153, 2072, 1408, 4), (100, 32700, 128, 0)])
def test_gemm_blocks(pkg, dev, M, N, K, Hv):
    test_gemm_kernel_edges(pkg, dev, M, N, K, Hv)


# Either side of the 8-wave kernel's lines: 132 tiles of 256 rows and 165 of 192
# (one round of 192 rows) at K of 2, 14 and 16 steps; 165 and 231 at 14 and 16
# steps; 260 tiles of 64 x 128 against 130 blocks at 24 and 26 steps, 195 against
# 130 (half empty blocks).  Whole tiles with a tail of quarters at K of 2 steps.
# The ring's 64-row tiles: 1024 rows, 4 MiB of A and more, one column block.
@pytest.mark.parametrize("M,N,K,Hv", [(900, 8224, 128, 16), (900, 8224, 896, 0), (900, 8224, 1024, 16),
                                      (1200, 8224, 896, 0), (1200, 8224, 1024, 4), (256, 8224, 1536, 16),
                                      (256, 8224, 1664, 16), (129, 8224, 1664, 0), (4100, 4008, 128, 4),
                                      (1024, 500, 1088, 4), (1500, 200, 1344, 4), (1500, 200, 1408, 0),
                                      (9000, 24, 1024, 0)])
def test_gemm_kernel_choice(pkg, dev, M, N, K, Hv):
    test_gemm_kernel_edges(pkg, dev, M, N, K, Hv)


def test_gemm_rows_do_not_depend_on_the_batch(pkg, dev):
    """64 x 128 tiles, 128 x 128 blocks, 192-row tiles and 256 x 256 tiles with a
    tail add a row's products in the same order: the same bits for the same rows."""
    gen = torch.Generator().manual_seed(8)
    x = torch.randn(2500, 1280, generator=gen).to(BF16).to(dev)
    w = (torch.randn(8224, 1280, generator=gen) / 36).to(BF16).to(dev)
    c = pkg.ops.linear(x, w)
    for M in (129, 300, 900):
        assert torch.equal(pkg.ops.linear(x[:M], w).view(torch.int16), c[:M].view(torch.int16)), M


@pytest.mark.parametrize("pad,off", [(40, 8), (41, 3)])
def test_gemm_strided_operands_and_out(pkg, dev, pad, off):
    """Row strides larger than K (views of wider buffers) and an output view;
    pad 41 / offset 3 gives an output row stride that is not a multiple of 4
    and rows at 2-byte alignment (element-by-element stores)."""
    gen = torch.Generator().manual_seed(5)
    M, N, K = 333, 264, 256
    abuf = torch.randn(M, K + 64, generator=gen).to(BF16)
    wbuf = (torch.randn(N, K + 128, generator=gen) / 16).to(BF16)
    a, w = abuf[:, 32:32 + K], wbuf[:, :K]
    out = torch.zeros(M, N + pad, dtype=BF16, device=dev)
    pkg.ops.linear(abuf.to(dev)[:, 32:32 + K], wbuf.to(dev)[:, :K], out=out[:, off:off + N])
    _check(out[:, off:off + N], *_ref(a, w), "strided gemm")
    assert torch.equal(out[:, :off].cpu(), torch.zeros(M, off, dtype=BF16))
    assert torch.equal(out[:, off + N:].cpu(), torch.zeros(M, pad - off, dtype=BF16))


@pytest.mark.parametrize("M", [100, 777, 1790])
def test_in_proj_with_gate_epilogue(pkg, dev, M):
    """The layer's in_proj over [W_qkv; W_z; W_b; W_a] (config 1 widths, a
    2048 hidden size): the projections, and g / beta from the b and a columns
    equal to fused_g_beta on them.  M = 100 runs 64 x 128 tiles, M = 777
    192 x 256 tiles, M = 1790 (231 tiles of 256 rows, 330 of 192) 256 x 256
    tiles."""
    gen = torch.Generator().manual_seed(6)
    Hk = Hv = 16
    D, hidden = 128, 2048
    C = 2 * Hk * D + Hv * D
    N = C + Hv * D + 2 * Hv
    x = torch.randn(M, hidden, generator=gen).to(BF16)
    w = (torch.randn(N, hidden, generator=gen) / math.sqrt(hidden)).to(BF16)
    A_log = (torch.rand(Hv, generator=gen) * math.log(16)).to(BF16)
    dt_bias = (torch.rand(Hv, generator=gen) * 2 - 1).to(BF16)
    y, g, beta = pkg.ops.linear(x.to(dev), w.to(dev), gates={"gate_col": C + Hv * D, "A_log": A_log.to(dev),
                                                             "dt_bias": dt_bias.to(dev)})
    _check(y, *_ref(x, w), "in_proj")
    b = y[:, C + Hv * D:C + Hv * D + Hv].contiguous()
    a = y[:, C + Hv * D + Hv:].contiguous()
    g2, beta2 = pkg.ops.fused_g_beta(b, a, A_log.to(dev), dt_bias.to(dev), None)
    torch.cuda.synchronize()
    assert torch.equal(g, g2) and torch.equal(beta.view(torch.int16), beta2.view(torch.int16))


def _layouts(C, V, Hv):
    # (the layer's three- and four-part in_proj; boundaries off the 32-column
    # grid, where one 32-column block's pieces go to two parts)
    return {"3": [C, V, 2 * Hv], "4": [C, V, Hv, Hv], "16": [48, C - 48, V + 16, 2 * Hv - 16]}


@pytest.mark.parametrize("layout", ["3", "4", "16"])
@pytest.mark.parametrize("with_gates", [False, True])
@pytest.mark.parametrize("M", [64, 100, 777, 1790])
def test_in_proj_column_parts_equal_one_output(pkg, dev, M, with_gates, layout):
    """gdn_gemm_bf16_cols (the layer's in_proj into separate qkv, z, b and a
    tensors): every part bit-equal to the same columns of the one-output GEMM,
    and the gate outputs too, for each tile shape (M = 64: 64 x 64 tiles with
    the deeper pipeline, 100: 64 x 128, 777: 256 x 256, 1790: 256 x 256 with a
    tail of quarters)."""
    gen = torch.Generator().manual_seed(7)
    Hk, Hv = 16, 32
    D, hidden = 128, 2048
    C = 2 * Hk * D + Hv * D
    V = Hv * D
    N = C + V + 2 * Hv
    x = torch.randn(M, hidden, generator=gen).to(BF16).to(dev)
    w = (torch.randn(N, hidden, generator=gen) / math.sqrt(hidden)).to(BF16).to(dev)
    A_log = (torch.rand(Hv, generator=gen) * math.log(16)).to(BF16).to(dev)
    dt_bias = (torch.rand(Hv, generator=gen) * 2 - 1).to(BF16).to(dev)
    gates = {"gate_col": C + V, "A_log": A_log, "dt_bias": dt_bias} if with_gates else None
    widths = _layouts(C, V, Hv)[layout]
    one = pkg.ops.linear(x, w, gates=gates)
    parts = pkg.ops.linear_cols(x, w, widths, gates=gates)
    torch.cuda.synchronize()
    if with_gates:
        (y, g, beta), (ps, g2, beta2) = one, parts
        assert torch.equal(g, g2) and torch.equal(beta.view(torch.int16), beta2.view(torch.int16))
    else:
        y, ps = one, parts
    c0 = 0
    for p, wd in zip(ps, widths):
        assert p.is_contiguous() and p.shape == (M, wd)
        assert torch.equal(p.view(torch.int16), y[:, c0:c0 + wd].contiguous().view(torch.int16)), (c0, wd)
        c0 += wd


def test_column_parts_rejected_shapes(pkg, dev):
    """Part boundaries off the 16-column grid, out of order, a last boundary
    other than N, or more than four parts are rejected before any launch.
    Real (small) buffers, each part's wide enough for every column, so even a
    launch that the checks had wrongly let through would stay in bounds."""
    import ctypes
    lib = pkg._lib.load()
    _lib = pkg._lib
    M, N, K = 4, 96, 64
    a = torch.zeros(M, K, dtype=BF16, device=dev)
    b = torch.zeros(N, K, dtype=BF16, device=dev)
    outs = [torch.zeros(M, 128, dtype=BF16, device=dev) for _ in range(5)]
    c = (ctypes.c_void_p * 5)(*[o.data_ptr() for o in outs])
    ld = (ctypes.c_int64 * 5)(*([128] * 5))
    stream = torch.cuda.current_stream(dev).cuda_stream

    def call(ends):
        e = (ctypes.c_int * len(ends))(*ends)
        return lib.gdn_gemm_bf16_cols(a.data_ptr(), K, b.data_ptr(), K, M, N, K, len(ends), c, ld, e, None, None,
                                      None, None, 0, 0, 0, stream)

    for ends in ((40, 96), (64, 100), (96, 64), (64, 64), (16, 32, 48, 64, 96), (8, 48, 64, 96)):
        assert call(ends) == _lib.GDN_ERR_INVALID_ARG, ends
    for ends in ((64, 96), (16, 48, 64, 96)):
        assert call(ends) == _lib.GDN_OK, ends
    torch.cuda.synchronize()
