"""The GatedDeltaNet prefill front (conv + SiLU, l2norm, gates, conv ring) in plain torch
(MI355X only)."""
import pytest
import torch

from qwen35_amd import abi

from _util import bf, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def at(t, off):
    """t on the GPU, its data off elements past an aligned address."""
    flat = torch.empty(t.numel() + off, dtype=t.dtype, device=DEV)[off:]
    flat.copy_(t.reshape(-1))
    return flat.view(t.shape)


def front(mixed, ring, conv_w, a, b, A_log, dt_bias, Hk, Hv, past, off=None):
    """off: the one buffer of mixed, conv_w, ring, y, qn, kn that is not 16-byte aligned."""
    M, C = mixed.shape
    d = [at(t, int(n == off)) for n, t in (("mixed", mixed), ("ring", ring), ("conv_w", conv_w), ("", a), ("", b),
                                           ("", A_log), ("", dt_bias))]
    y, qn, kn = (at(torch.zeros(M, c, dtype=torch.bfloat16), int(n == off))
                 for n, c in (("y", C), ("qn", Hk * 128), ("kn", Hk * 128)))
    g, beta = torch.empty(M, Hv, device=DEV), torch.empty(M, Hv, dtype=torch.bfloat16, device=DEV)
    p = abi.ptr
    abi.check(abi.load().qh_gdn_prep(*[p(t) for t in d], p(y), p(qn), p(kn), p(g), p(beta), M, Hk, Hv, 128, 128, past,
                                     abi.stream_handle()), "gdn_prep")
    torch.cuda.synchronize()
    return [t.cpu() for t in (y, qn, kn, g, beta, d[1])]


# 1 token per thread, 16 per block; the ring holds the last four positions, so prompts of fewer than 4 tokens keep some of its old ones.
# With one buffer 2 bytes past a 16-byte boundary the conv and the norm run as two kernels.
@pytest.mark.parametrize("M,past,off", [(1, 0, None), (1, 6, None), (2, 3, None), (3, 9, None), (4, 1, None),
                                        (5, 2, None), (31, 0, None), (33, 7, None), (511, 5, None), (512, 0, None),
                                        (513, 6, None), (700, 3, None), (1, 6, "mixed"), (3, 9, "ring"),
                                        (5, 2, "conv_w"), (33, 7, "y"), (513, 6, "qn"), (40, 0, "kn")])
def test_gdn_front(M, past, off):
    Hk, Hv = 2, 4
    C = (2 * Hk + Hv) * 128
    g = gen(M + past)
    mixed, ring = bf(randn(g, M, C)), bf(randn(g, C, 4))
    w, a, b = bf(randn(g, C, 4, std=0.5)), bf(randn(g, M, Hv)), bf(randn(g, M, Hv))
    A_log, dt = randn(g, Hv), randn(g, Hv)
    y, qn, kn, gl, beta, r2 = front(mixed, ring, w, a, b, A_log, dt, Hk, Hv, past, off)
    before = torch.stack([ring[:, (past + t) % 4] for t in (-3, -2, -1)])
    x = torch.cat([before, mixed]).double()
    acc = sum(x[j:j + M] * w.double()[:, j] for j in range(4))
    ref = torch.nn.functional.silu(acc.float().to(torch.bfloat16).double())
    # one flip of the conv's bf16 rounding (2^-7 of it), where silu's slope is at most 1.1, and the result's own
    assert ((y.double() - ref).abs() <= 1.1 * 2.0 ** -7 * acc.abs() + 2.0 ** -8 * ref.abs() + 1e-30).all()
    for got, c0 in ((qn, 0), (kn, Hk * 128)):
        v = y[:, c0:c0 + Hk * 128].double().view(M, Hk, 128)
        n = (v * torch.rsqrt((v * v).sum(-1, keepdim=True) + 1e-6)).view(M, -1)
        # bf16 steps: the squares, the sum, the reciprocal root and the product
        assert ((got.double() - n).abs() <= 3 * 2.0 ** -8 * n.abs() + 1e-30).all()
    assert torch.allclose(gl.double(), -torch.exp(A_log.double()) * torch.nn.functional.softplus(a.double() + dt.double()),
                          rtol=1e-5, atol=1e-30)
    assert ((beta.double() - torch.sigmoid(b.double())).abs() <= 2.0 ** -8).all()
    want = ring.clone()
    for t in range(max(0, M - 4), M):
        want[:, (past + t) % 4] = mixed[t]
    assert torch.equal(r2, want)


@pytest.mark.parametrize("M", [176, 683])
def test_conv_silu_every_argument(M):
    """Every finite bf16 value through a conv that passes its newest token: rounded as 64-bit SiLU at
    least as often as fp32 arithmetic is, and never more than one bf16 step off; infinities."""
    C = 3 * 128
    allv = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    fin = allv[torch.isfinite(allv.float())]
    x = torch.zeros(M * C, dtype=torch.bfloat16)
    x[:fin.numel()] = fin
    x = x.view(M, C)
    w = torch.zeros(C, 4, dtype=torch.bfloat16)
    w[:, 3] = 1.0
    z = torch.zeros(M, 1, dtype=torch.bfloat16)
    y = front(x, torch.zeros(C, 4, dtype=torch.bfloat16), w, z, z, torch.zeros(1), torch.zeros(1), 1, 1, 0)[0].float()
    exact = (x.double() / (1 + torch.exp(-x.double()))).float().to(torch.bfloat16).float()
    f32 = (x.float() / (1 + torch.exp(-x.float()))).to(torch.bfloat16).float()
    normal = exact.abs() > 1e-36
    assert int((y != exact)[normal].sum()) <= int((f32 != exact)[normal].sum())
    assert ((y - exact).abs() <= 2.0 ** -7 * exact.abs() + 1e-36).all()
    # the lower end, where e^-x nears the largest fp32 number: normal results down to -88.5, zero below as
    # in fp32 (1 + e^-x is infinite there)
    low = x.float() <= -87.0
    assert int((f32[low] != 0).sum()) >= 4 and ((y - f32).abs() <= 2.0 ** -7 * f32.abs())[low].all()
    x = torch.zeros(M, C, dtype=torch.bfloat16)
    x[-1, :3] = torch.tensor([float("inf"), -float("inf"), float("nan")])
    y = front(x, torch.zeros(C, 4, dtype=torch.bfloat16), w, z, z, torch.zeros(1), torch.zeros(1), 1, 1, 0)[0].float()
    assert y[-1, 0] == float("inf") and torch.isnan(y[-1, 1:3]).all()


@pytest.mark.parametrize("off", ["out", "z", "norm_w"])
@pytest.mark.parametrize("M", [1, 9, 70])
def test_gated_norm_unaligned(M, off):
    """The gated norm after the scan with one operand 2 bytes past a 16-byte boundary (an element per
    thread) against the 16-byte kernel: the same scan output, whose sum of squares is added in another
    order, so that each of three bf16 roundings may fall to the other side (2^-8 of the value each)."""
    Hk, Hv = 2, 4
    g = gen(M)
    bf16 = [bf(randn(g, M, Hk * 128)), bf(randn(g, M, Hk * 128)), bf(randn(g, M, (2 * Hk + Hv) * 128))]
    gl, beta = -torch.rand(M, Hv, generator=g), bf(torch.rand(M, Hv, generator=g))
    z, nw, state = bf(randn(g, M, Hv * 128)), bf(1 + randn(g, 128, std=0.02)), randn(g, Hv, 128, 128, std=0.1)
    res = []
    for o in (None, off):
        q, k, y = (at(t, 0) for t in bf16)
        dg, db, dz, dn, ds = at(gl, 0), at(beta, 0), at(z, int(o == "z")), at(nw, int(o == "norm_w")), at(state, 0)
        out = at(torch.zeros(M, Hv * 128, dtype=torch.bfloat16), int(o == "out"))
        p = abi.ptr
        abi.check(abi.load().qh_gdn_scan(p(q), p(k), p(y), p(dg), p(db), p(dz), p(dn), p(ds), p(out), M, Hk, Hv, 128,
                                         128, 1e-6, abi.stream_handle()), "gdn_scan")
        torch.cuda.synchronize()
        res.append((out.float().cpu(), ds.cpu()))
    (a, sa), (b, sb) = res
    assert torch.equal(sa, sb) and a.abs().max() > 0
    assert ((a - b).abs() <= 3 * 2.0 ** -8 * a.abs() + 1e-30).all()
