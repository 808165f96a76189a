"""Shared helpers for the parity tests."""
import ctypes

import torch

from oracle import qwen35_oracle as orc


def gen(seed=0):
    g = torch.Generator()
    g.manual_seed(seed)
    return g


def randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g) * std


def bf(x):
    return x.to(torch.bfloat16)


def cos_sim(a, b):
    a = a.double().reshape(-1)
    b = b.double().reshape(-1)
    return float((a @ b) / (a.norm() * b.norm() + 1e-300))


def assert_close(got, ref, rtol=1e-2, atol_frac=1e-4, min_cos=0.99999, what=""):
    """bf16-output parity: |got - ref| <= rtol*|ref| + atol_frac*max|ref|
    elementwise, and cosine similarity >= min_cos."""
    got = got.detach().float().cpu().reshape(-1)
    ref = ref.detach().float().cpu().reshape(-1)
    assert got.shape == ref.shape, (what, got.shape, ref.shape)
    assert torch.isfinite(got).all(), f"{what}: non-finite output"
    tol = rtol * ref.abs() + atol_frac * ref.abs().max()
    bad = (got - ref).abs() > tol
    nbad = int(bad.sum())
    c = cos_sim(got, ref)
    if nbad or c < min_cos:
        i = int(((got - ref).abs() - tol).argmax())
        raise AssertionError(f"{what}: {nbad}/{ref.numel()} outside tolerance, cos={c:.8f}; "
                             f"worst i={i} got={got[i].item():.6g} ref={ref[i].item():.6g}")
    return c


def quant(g, n, k, std=0.02):
    return orc.quantize_block_fp8(randn(g, n, k, std=std))


def gemm_plan(M, K, N, ws=None, kb=None, cus=256):
    """qh_gemm_plan by field names; ws None: a workspace of the full size."""
    from qwen35_amd import abi
    lib, out = abi.load(), (ctypes.c_int * 7)()
    if ws is None:
        ws = int(lib.qh_gemm_workspace_size(M, K))
    abi.check(lib.qh_gemm_plan(M, K, len(N), ctypes.cast((ctypes.c_int * len(N))(*N), ctypes.c_void_p),
                               K // 128 if kb is None else kb, cus, ws, ctypes.cast(out, ctypes.c_void_p)), "plan")
    return dict(zip(("tile", "bm", "bn", "wpc", "nstep", "S", "load"), out))


def gemm_shape(M, K, N, ws=None, cus=256):
    """The shape a product runs on, "t3" (tile kernel) or "r128" (ring kernel, columns of its tile), with
    its K slices where there are several: "t3/4"."""
    p = gemm_plan(M, K, N, ws, cus=cus)
    name = f"t{p['tile']}" if p["tile"] >= 0 else f"r{p['bn']}"
    return name if p["S"] == 1 else f"{name}/{p['S']}"
