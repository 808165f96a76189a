"""The GatedDeltaNet prefill front (conv + SiLU, l2norm, gates, conv ring) in plain torch
(MI355X only)."""
import pytest
import torch

from qwen35_amd import abi

from _util import bf, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def front(mixed, ring, conv_w, a, b, A_log, dt_bias, Hk, Hv, past):
    M, C = mixed.shape
    d = [t.to(DEV).contiguous() for t in (mixed, ring, conv_w, a, b, A_log, dt_bias)]
    bfo = dict(dtype=torch.bfloat16, device=DEV)
    y, qn, kn = torch.empty(M, C, **bfo), torch.empty(M, Hk * 128, **bfo), torch.empty(M, Hk * 128, **bfo)
    g, beta = torch.empty(M, Hv, device=DEV), torch.empty(M, Hv, **bfo)
    p = abi.ptr
    abi.check(abi.load().qh_gdn_prep(*[p(t) for t in d], p(y), p(qn), p(kn), p(g), p(beta), M, Hk, Hv, 128, 128, past,
                                     abi.stream_handle()), "gdn_prep")
    torch.cuda.synchronize()
    return [t.cpu() for t in (y, qn, kn, g, beta, d[1])]


# 1 token per thread (16 per block) below 512 tokens, 8 (128 per block) from there; the ring holds
# the last four positions, so prompts of fewer than 4 tokens keep some of its old ones.
@pytest.mark.parametrize("M,past", [(1, 0), (1, 6), (2, 3), (3, 9), (4, 1), (5, 2), (31, 0), (33, 7), (511, 5),
                                    (512, 0), (513, 6), (700, 3)])
def test_gdn_front(M, past):
    Hk, Hv = 2, 4
    C = (2 * Hk + Hv) * 128
    g = gen(M + past)
    mixed, ring = bf(randn(g, M, C)), bf(randn(g, C, 4))
    w, a, b = bf(randn(g, C, 4, std=0.5)), bf(randn(g, M, Hv)), bf(randn(g, M, Hv))
    A_log, dt = randn(g, Hv), randn(g, Hv)
    y, qn, kn, gl, beta, r2 = front(mixed, ring, w, a, b, A_log, dt, Hk, Hv, past)
    before = torch.stack([ring[:, (past + t) % 4] for t in (-3, -2, -1)])
    x = torch.cat([before, mixed]).double()
    acc = sum(x[j:j + M] * w.double()[:, j] for j in range(4))
    ref = torch.nn.functional.silu(acc.float().to(torch.bfloat16).double())
    # one flip of the conv's bf16 rounding (2^-7 of it), where silu's slope is at most 1.1, and the result's own
    assert ((y.double() - ref).abs() <= 1.1 * 2.0 ** -7 * acc.abs() + 2.0 ** -8 * ref.abs() + 1e-30).all()
    for got, at in ((qn, 0), (kn, Hk * 128)):
        v = y[:, at:at + Hk * 128].double().view(M, Hk, 128)
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


@pytest.mark.parametrize("M", [176, 683])   # both thread shapes
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
