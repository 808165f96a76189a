"""The prefill GEMM's tile shapes against the product in 64 bits (MI355X only)."""
import pytest
import torch

from oracle import qwen35_oracle as orc
from qwen35_amd import abi, ops

from _util import bf, gemm_shape, gen, quant, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def product(x, w, s):
    """(X deq(W)^T, |X| |deq(W)|^T) in 64 bits."""
    d = orc.dequant(w, s.float()).to(DEV).double()
    x = x.to(DEV).double()
    return x @ d.t(), x.abs() @ d.abs().t()


def check(y, ref, mag, K, what):
    """bf16 rounding of the result (8 significant bits: at most 2^-8 of it) and K fp32 additions of products
    whose magnitudes add up to mag (each at most 2^-24 of a partial sum <= mag)."""
    err = (y.double() - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + mag * (K * 2.0 ** -24) + 1e-38
    bad = err > bound
    assert torch.isfinite(y.float()).all() and not bad.any(), \
        f"{what}: {int(bad.sum())} of {bad.numel()} off, worst {float((err / bound).max()):.2f} of the bound"


def shape_is(M, K, N, ws, want):
    """The plan takes the shape that a row is meant for (rows are chosen for 256 CUs)."""
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert gemm_shape(M, K, N, ws) == want


# The shape that 256 CUs take for each (rows x columns of the tile, waves along K), at row and
# column counts that leave ragged last tiles; K is as short as the shape's choice allows, so that
# K groups with no unit of their own and rings longer than K are among them.
SHAPES = {
    "t0": [(2, 4, 256), (9, 5, 640), (16, 2560, 9216), (17, 33, 256)],              # 16 x 16, 8 waves
    "t1": [(2, 8544, 384), (3, 8217, 640), (16, 9999, 2560), (2, 9301, 896)],       # 16 x 48, 8 waves
    "t2": [(2, 4185, 256), (31, 2561, 4096), (65, 1673, 256)],                      # 32 x 32, 8 waves
    "t3": [(29, 9030, 512), (72, 2827, 384)],                                       # 32 x 48, 8 waves
    "t4": [(33, 6549, 768), (91, 4315, 896), (131, 2522, 768)],                     # 64 x 48, 4 waves
    "t5": [(271, 2523, 1024), (2, 12435, 768), (24, 18159, 1024)],                  # 32 x 160, 2 groups
    "t6": [(329, 5681, 2560), (262, 6697, 1536), (2288, 540, 256)],                 # 64 x 160, 2 groups
    "t7": [(2490, 1595, 384), (736, 6687, 384), (1030, 3171, 1024)],                # 128 x 160
    "t8": [(603, 12393, 512), (900, 14615, 1280), (2333, 2272, 256)],               # 128 x 256
    "t9": [(412, 18795, 1280), (1190, 6551, 1536), (2665, 3138, 768)],              # 128 x 320
    "r64": [(71, 15113, 256), (866, 1779, 256), (129, 9217, 1536), (2, 16557, 256), (5, 300, 16512)],
    "r128": [(137, 13615, 256), (389, 18401, 2560), (448, 18432, 2560), (943, 8514, 384)],
    "r192": [(755, 7201, 1024), (1796, 2875, 768)],
}


@pytest.mark.parametrize("shape,M,N,K", [(k, *v) for k, vs in SHAPES.items() for v in vs] + [("t0", 5, 300, 16384)])
def test_gemm_tile_shapes(shape, M, N, K):
    shape_is(M, K, (N,), 0, shape)
    g = gen(M * 3 + N + K)
    w, s = quant(g, N, K)
    s = s * (1.0 + torch.rand(s.shape, generator=g))   # scales that differ from block to block
    s[-1, -1] = 0.0                                    # and an empty block
    x = bf(randn(g, M, K))
    for scale in (s, s.to(torch.bfloat16)):            # bf16: fp8_gemm_batch
        ref, mag = product(x, w, scale)
        y = ops.fp8_linear(x.to(DEV), w.to(DEV), scale.to(DEV))
        check(y, ref, mag, K, f"{M} x {N} x {K} {scale.dtype}")


# Rows that are not 8-byte aligned: every residue of the row stride mod 4, the first element on an
# odd and on an even 2-byte address, last tiles of one column, an odd and an even number of them.
# The elements before and after the output stay as they were.
@pytest.mark.parametrize("shape,M,N,K", [("t5", 2, 18621, 1024), ("t5", 36, 13581, 1280), ("t5", 3, 18698, 896),
                                         ("t6", 783, 2529, 1024), ("t6", 2201, 706, 896), ("t7", 579, 6201, 512),
                                         ("t7", 203, 16581, 512), ("t7", 403, 9754, 512), ("t8", 458, 15373, 1280),
                                         ("t8", 603, 12393, 512), ("t8", 1666, 4246, 384), ("t9", 731, 11477, 896),
                                         ("t9", 2613, 3426, 512), ("t0", 2, 1, 256), ("t2", 5, 4185, 256)])
@pytest.mark.parametrize("off", [0, 1, 2])
def test_gemm_tile_unaligned_rows(shape, M, N, K, off):
    shape_is(M, K, (N,), 0, shape)
    g = gen(M + N + off)
    w, s = quant(g, N, K)
    x, dw, ds = bf(randn(g, M, K)), w.to(DEV), s.to(DEV)
    buf = torch.full((M * N + 16,), 77.0, dtype=torch.bfloat16, device=DEV)
    y, dx, lib = buf[off:off + M * N], x.to(DEV), abi.load()
    abi.check(lib.qh_gemm_e4m3(abi.ptr(dx), abi.ptr(dw), abi.ptr(ds), abi.ptr(y), M, N, K, K // 128, 0, None, 0,
                               abi.stream_handle()), "gemm")
    check(y.view(M, N), *product(x, w, s), K, f"{M} x {N} x {K} at {off}")
    assert (buf[:off] == 77.0).all() and (buf[off + M * N:] == 77.0).all()


@pytest.mark.parametrize("shape,M,N,K", [
    ("t3/2", 100, 840, 5120), ("t3/4", 24, 2560, 9216), ("t3/8", 20, 53, 5120), ("t4/2", 630, 538, 9216),
    ("t4/4", 33, 2560, 9216), ("t4/8", 37, 1001, 9216), ("t5/2", 2, 12563, 1024), ("t5/8", 16, 4380, 6144),
    ("t6/2", 512, 2560, 9216), ("t6/4", 224, 2560, 9216), ("t6/8", 128, 2560, 9216), ("t7/8", 317, 1586, 9216),
    ("r64/2", 300, 2560, 2560), ("r64/3", 143, 3469, 3072), ("r64/4", 150, 2560, 4096), ("r64/6", 48, 4249, 3072),
    ("r128/2", 600, 2560, 9216), ("r128/4", 300, 2560, 9216), ("r128/5", 220, 3018, 5120)])
def test_gemm_tile_split_k(shape, M, N, K):
    """K slices over workgroups (a workspace given), plain and fused with the residual add."""
    shape_is(M, K, (N,), None, shape)
    g = gen(M + N + K)
    w, s = quant(g, N, K)
    x, h = bf(randn(g, M, K)).to(DEV), bf(randn(g, M, N)).to(DEV)
    lib = abi.load()
    dw, ds = w.to(DEV), s.to(DEV)
    ws = torch.full((int(lib.qh_gemm_workspace_size(M, K)),), 0xFF, dtype=torch.uint8, device=DEV)  # NaN partials
    y, o = torch.empty(2, M, N, dtype=torch.bfloat16, device=DEV).unbind(0)
    abi.check(lib.qh_gemm_e4m3(abi.ptr(x), abi.ptr(dw), abi.ptr(ds), abi.ptr(y), M, N, K, K // 128, 0, abi.ptr(ws),
                               ws.numel(), abi.stream_handle()), "gemm")
    ref, mag = product(x, w, s)
    check(y, ref, mag, K, "workspace")
    h2 = h.clone()
    abi.check(lib.qh_gemm_e4m3_add_rmsnorm(abi.ptr(x), abi.ptr(dw), abi.ptr(ds), abi.ptr(o), M, N, K, K // 128, 0,
                                           abi.ptr(h2), None, None, 1e-6, abi.ptr(ws), ws.numel(),
                                           abi.stream_handle()), "gemm_add")
    assert torch.equal(h2, (h.float() + y.float()).to(torch.bfloat16))


@pytest.mark.parametrize("M", [3, 20, 128, 700])
def test_gemm_tile_segments(M):
    """Segments of unequal width, one of them a few columns, each with its own scales."""
    K, ns = 1024, (1000, 8192, 32, 5)
    g = gen(M)
    x = bf(randn(g, M, K))
    dx, lib = x.to(DEV), abi.load()
    segs = [quant(g, n, K) for n in ns]
    ys = [torch.empty(M, n, dtype=torch.bfloat16, device=DEV) for n in ns]
    keep, args = [], []
    for (w, s), y, n in zip(segs, ys, ns):
        keep += [w.to(DEV), s.to(DEV)]
        args += [abi.ptr(keep[-2]), abi.ptr(keep[-1]), abi.ptr(y), n, K // 128]
    abi.check(lib.qh_gemm_e4m3_grouped(abi.ptr(dx), M, K, 4, *args, 0, None, 0, abi.stream_handle()), "grouped")
    for (w, s), y, n in zip(segs, ys, ns):
        check(y, *product(x, w, s), K, f"{M} rows, {n} columns")


@pytest.mark.parametrize("shape,M,ns,K", [
    ("t5/2", 2, (7247, 2258, 34, 7689), 2560), ("t5/2", 17, (7614, 5230, 1164, 4731), 3072),
    ("t6/2", 33, (9216, 9216), 2560), ("t6/2", 172, (43, 4193, 304, 938), 4096), ("t6/2", 234, (548, 4093), 4096),
    ("r64/2", 102, (4314, 3533, 57), 3072), ("r128/4", 73, (1113, 5862), 3072)])
def test_gemm_segments_split_k(shape, M, ns, K):
    """K slices of several segments, which end inside tiles, finished by the reduction kernel; a workspace of NaN."""
    shape_is(M, K, ns, None, shape)
    g = gen(M + K)
    x = bf(randn(g, M, K))
    dx, lib = x.to(DEV), abi.load()
    segs = [quant(g, n, K) for n in ns]
    ys = [torch.empty(M, n, dtype=torch.bfloat16, device=DEV) for n in ns]
    ws = torch.full((int(lib.qh_gemm_workspace_size(M, K)),), 0xFF, dtype=torch.uint8, device=DEV)
    keep, args = [], []
    for (w, s), y, n in zip(segs, ys, ns):
        keep += [w.to(DEV), s.to(DEV)]
        args += [abi.ptr(keep[-2]), abi.ptr(keep[-1]), abi.ptr(y), n, K // 128]
    args += [None, None, None, 0, 0] * (4 - len(ns))
    abi.check(lib.qh_gemm_e4m3_grouped(abi.ptr(dx), M, K, len(ns), *args, 0, abi.ptr(ws), ws.numel(),
                                       abi.stream_handle()), "grouped")
    for (w, s), y, n in zip(segs, ys, ns):
        check(y, *product(x, w, s), K, f"{M} rows, {n} columns")


@pytest.mark.parametrize("M,N,K", [(1, 100, 64), (2, 1003, 256), (32, 260, 2560), (33, 1001, 192), (64, 4096, 256),
                                   (65, 130, 320), (129, 1027, 2560), (300, 520, 128)])
def test_lm_head_rows(M, N, K):
    """Row blocks of 32, 64 and 128 by 128 columns with ragged ends; a row's logits are the same
    bits however many rows come with it."""
    g = gen(M + N + K)
    x, w, nw = bf(randn(g, M, K)).to(DEV), bf(randn(g, N, K, std=0.02)).to(DEV), randn(g, K, std=0.02).to(DEV)
    lib = abi.load()
    xn, ref_xn = torch.empty(2, M, K, dtype=torch.bfloat16, device=DEV).unbind(0)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)

    def run(xx, yy, m):
        abi.check(lib.qh_lm_head_rows(abi.ptr(xx), abi.ptr(nw), 1e-6, m, K, abi.ptr(w), N, abi.ptr(xn), abi.ptr(yy),
                                      abi.stream_handle()), "lm_head_rows")
    run(x, y, M)
    abi.check(lib.qh_rmsnorm(abi.ptr(x), abi.ptr(nw), abi.ptr(ref_xn), M, K, 1e-6, abi.stream_handle()), "rmsnorm")
    assert torch.equal(xn, ref_xn)
    d, dw = xn.double(), w.double()
    check(y, d @ dw.t(), d.abs() @ dw.abs().t(), K, "lm_head rows")
    last = torch.empty(1, N, dtype=torch.bfloat16, device=DEV)
    run(x[M - 1:].contiguous(), last, 1)
    assert torch.equal(last[0], y[M - 1])
