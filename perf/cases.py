"""The work a user of this framework has it do, as cases that can be timed and compared.

Each case is a dict of plain values; `kind` names the path it goes through:

  linear       one E4M3 projection, `ops.fp8_linear` (M = 1: decode GEMV, else the prefill GEMM)
  mlp_decode   one decode token's MLP block, `qh_mlp_decode`
  mlp          a prompt's MLP block: gate and up in one grouped GEMM, SiLU * up, down with the
               residual add and the norm that follows it
  attn_decode  one decode token's attention mixer over a KV cache, `qh_attn_decode`
  attn         a prompt's attention mixer: head norms, RoPE and cache write, then causal attention
  gdn          a prompt's GatedDeltaNet mixer: conv and gates, then the delta rule and gated norm
  chat         engine: a prompt's batch prefill, then decode steps by the captured graph
  score        engine: the logits of every position of a text (logits_to_keep = 0)

Shapes are those of the 4B model that `config.qwen35_4b` describes (hidden 2560, intermediate
9216, 16 / 4 attention heads of 256, 16 / 32 GatedDeltaNet heads of 128, vocabulary 248320).  The
whole-model cases run one period of its layer pattern (three GatedDeltaNet layers and one
attention layer) with the full embedding and head: a change of rounding in one layer travels
through all that follow, so that the 32 layers of a random-weight model say nothing about the
outputs any more.
"""
import math

import torch

import __graft_entry__

__graft_entry__.load_package()

from qwen35_amd import abi, engine, ops, synth  # noqa: E402
from qwen35_amd.config import Qwen35Config  # noqa: E402

DEV = "cuda"
BF = torch.bfloat16
CFG = Qwen35Config(num_hidden_layers=4)
H, I, V = CFG.hidden_size, CFG.intermediate_size, CFG.vocab_size
D, HQ, HKV, ROT = CFG.head_dim, CFG.num_attention_heads, CFG.num_key_value_heads, CFG.rotary_dim
HK, HV, DL = CFG.linear_num_key_heads, CFG.linear_num_value_heads, CFG.linear_key_head_dim
CONV = CFG.conv_dim
EPS = CFG.rms_norm_eps
MAX_SEQ = 4096
GDN_CHUNK_MIN = 96      # tokens from which a prompt's delta rule runs in the chunked form
STD = 0.02              # weight scale of the random models, as synth.make_weights


def listed():
    return [
        # one token's projection to the MLP width, the decode step's commonest size
        {"name": "linear_decode", "kind": "linear", "M": 1, "K": 2560, "N": 9216, "scale": "float32",
         "mode": "block"},
        # the down projection of a short chat turn continued on a cache
        {"name": "linear_turn", "kind": "linear", "M": 24, "K": 9216, "N": 2560, "scale": "bfloat16",
         "mode": "block"},
        # a half-thousand-token prompt through the reference's symbol (bf16 scales, no workspace)
        {"name": "linear_prompt", "kind": "linear", "M": 512, "K": 2560, "N": 9216, "scale": "bfloat16",
         "mode": "block"},
        # one token's MLP block
        {"name": "mlp_decode", "kind": "mlp_decode"},
        # the MLP block of an ordinary prompt and of a document near the cache's length
        {"name": "mlp_prompt", "kind": "mlp", "M": 128},
        {"name": "mlp_long", "kind": "mlp", "M": 3700},
        # one token's attention over a full cache
        {"name": "attn_decode", "kind": "attn_decode", "ctx": 4096},
        # a document's attention layer
        {"name": "attn_long", "kind": "attn", "M": 3700, "past": 0},
        # an ordinary prompt's and a document's GatedDeltaNet layer
        {"name": "gdn_prompt", "kind": "gdn", "M": 128},
        {"name": "gdn_long", "kind": "gdn", "M": 3700},
        # a text's logits at every position: what perplexity and choice scoring ask for
        {"name": "score", "kind": "score", "M": 96},
        # a prompt and the first tokens of the answer, teacher-forced so that every step's logits
        # can be compared
        {"name": "chat", "kind": "chat", "M": 128, "steps": 8},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "attn", "attn", "gdn", "gdn",
                       "attn_decode", "chat", "score"])
    if kind == "linear":
        # the model's projections, and row counts that fit no tile
        K, N = rng.choice([(2560, 9216), (9216, 2560), (4096, 2560), (2560, 8192), (2560, 4096),
                           (2560, 1024), (2560, 32), (256, 512), (2560, rng.randint(100, 9000)),
                           (128 * rng.randint(2, 72), rng.randint(33, 6000))])
        return {"kind": kind, "M": _log_int(rng, 1, 4096), "K": K, "N": N,
                "scale": rng.choice(["float32", "bfloat16"]), "mode": rng.choice(["block", "block", "block", "row"])}
    if kind in ("mlp", "gdn"):
        return {"kind": kind, "M": _log_int(rng, 2, 3700)}
    if kind == "attn":
        M = _log_int(rng, 2, 3700)
        return {"kind": kind, "M": M, "past": rng.choice([0, 0, rng.randint(1, MAX_SEQ - M)])}
    if kind == "attn_decode":
        return {"kind": kind, "ctx": _log_int(rng, 1, MAX_SEQ)}
    if kind == "chat":
        return {"kind": kind, "M": _log_int(rng, 2, 1000), "steps": rng.randint(1, 8)}
    return {"kind": kind, "M": _log_int(rng, 2, 96)}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _fp8(g, n, k, mode="block"):
    """(E4M3 bytes, fp32 scale_inv): 128 x 128 blocks as a checkpoint holds them, or one per row."""
    w = _randn(g, n, k) * STD
    if mode == "block":
        return synth.quantize_block_fp8(w)
    s = (w.abs().amax(1) / 448.0).clamp(min=1e-12)
    return (w / s[:, None]).to(torch.float8_e4m3fn).view(torch.uint8), s.contiguous()


def _inputs(case, seed):
    """What the seed alone determines, before any buffer of the framework's."""
    g, k = _gen(seed), case["kind"]
    if k == "linear":
        w, s = _fp8(g, case["N"], case["K"], case["mode"])
        return {"x": _randn(g, case["M"], case["K"]).to(BF), "w": w, "s": s.to(getattr(torch, case["scale"]))}
    if k in ("mlp", "mlp_decode"):
        M = case.get("M", 1)
        return {"h": _randn(g, M, H).to(BF), "x": _randn(g, M, H).to(BF), "norm": _randn(g, H) * STD,
                "gate": _fp8(g, I, H), "up": _fp8(g, I, H), "down": _fp8(g, H, I)}
    if k in ("attn", "attn_decode"):
        M, past = (case["M"], case["past"]) if k == "attn" else (1, case["ctx"] - 1)
        kc, vc = torch.zeros(2, HKV, MAX_SEQ, D, dtype=BF, device=DEV).unbind(0)
        kc[:, :past] = _randn(g, HKV, past, D).to(BF)
        vc[:, :past] = _randn(g, HKV, past, D).to(BF)
        cos, sin = engine.rope_tables(MAX_SEQ, ROT, CFG.rope_theta, device=DEV)
        return {"q": _randn(g, M, HQ, 2 * D).to(BF), "k": _randn(g, M, HKV, D).to(BF),
                "v": _randn(g, M, HKV, D).to(BF), "qn": _randn(g, D) * STD, "kn": _randn(g, D) * STD,
                "kc": kc, "vc": vc, "cos": cos, "sin": sin}
    if k == "gdn":
        M = case["M"]
        u = torch.rand(HV, generator=g, device=DEV)
        return {"mixed": _randn(g, M, CONV).to(BF), "z": _randn(g, M, HV, DL).to(BF), "a": _randn(g, M, HV).to(BF),
                "b": _randn(g, M, HV).to(BF), "conv_w": (_randn(g, CONV, 4) * 0.3).to(BF),
                "A_log": torch.log(1e-3 + u * (16.0 - 1e-3)), "dt_bias": torch.ones(HV, device=DEV),
                "norm": (1.0 + _randn(g, DL) * STD).to(BF)}
    raise ValueError(k)


def prepare(case, seed):
    k = case["kind"]
    if k in ("chat", "score"):
        M, n = case["M"], case["M"] + case.get("steps", 0)
        w = synth.make_weights(CFG, seed=seed, device=DEV)
        eng = engine.Qwen35FP8Engine(w, max_seq_len=MAX_SEQ)
        ids = synth.make_prompt(CFG, n=n, seed=seed + 1, device=DEV)
        if k == "chat":
            eng.capture()
        return {"case": case, "eng": eng, "prompt": ids[:M].view(1, -1), "next": [ids[t:t + 1].view(1, 1) for t in range(M, n)]}
    s = _inputs(case, seed)
    s.update(case=case, lib=abi.load())
    lib = s["lib"]

    def empty(*shape, dtype=BF):
        return torch.empty(*shape, dtype=dtype, device=DEV)

    if k == "mlp_decode":
        s.update(m=empty(I), out=empty(H))
    elif k == "mlp":
        M = case["M"]
        s.update(g=empty(M, I), u=empty(M, I), m=empty(M, I), o=empty(M, H), hn=empty(M, H),
                 ws=empty(int(lib.qh_gemm_workspace_size(M, I)), dtype=torch.uint8))
    elif k == "attn_decode":
        ns = engine.default_attn_splits(MAX_SEQ)
        s.update(splits=ns, out=empty(HQ * D),
                 scratch=torch.zeros(int(lib.qh_attn_scratch_bytes(HKV, ns, D)), dtype=torch.uint8, device=DEV),
                 counters=torch.zeros(HKV, dtype=torch.int32, device=DEV),
                 pos=torch.full((1,), case["ctx"] - 1, dtype=torch.int32, device=DEV))
    elif k == "attn":
        M = case["M"]
        s.update(q32=empty(M, HQ, D, dtype=torch.float32), out=empty(M, HQ * D))
    elif k == "gdn":
        M = case["M"]
        s.update(ring=empty(CONV, 4), y=empty(M, CONV), qn=empty(M, HK * DL), kn=empty(M, HK * DL),
                 g=empty(M, HV, dtype=torch.float32), beta=empty(M, HV), out=empty(M, HV * DL),
                 state=empty(HV, DL, DL, dtype=torch.float32),
                 ws=empty(max(int(lib.qh_gdn_chunk_workspace_size(M, HV)), 16), dtype=torch.uint8))
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    case = s["case"]
    k, p, st = case["kind"], abi.ptr, abi.stream_handle()
    if k == "linear":
        return ops.fp8_linear(s["x"], s["w"], s["s"])
    if k == "chat":
        eng = s["eng"]
        logits = [eng.forward(s["prompt"], 0).clone()]
        pos = s["prompt"].numel()
        for t, tok in enumerate(s["next"]):
            logits.append(eng.forward(tok, pos + t).clone())
        return logits
    if k == "score":
        return s["eng"].forward(s["prompt"], 0, logits_to_keep=0)
    L = s["lib"]
    if k == "mlp_decode":
        abi.check(L.qh_mlp_decode(p(s["h"]), p(s["x"]), p(s["norm"]), EPS, H, p(s["gate"][0]), p(s["gate"][1]),
                                  p(s["up"][0]), p(s["up"][1]), I, H // 128, p(s["down"][0]), p(s["down"][1]),
                                  I // 128, p(s["m"]), p(s["out"]), 0, st), "mlp_decode")
        return s["out"]
    if k == "mlp":
        M, ws = case["M"], s["ws"]
        none = (None, None, None, 0, 0)
        abi.check(L.qh_gemm_e4m3_grouped(p(s["x"]), M, H, 2, p(s["gate"][0]), p(s["gate"][1]), p(s["g"]), I, H // 128,
                                         p(s["up"][0]), p(s["up"][1]), p(s["u"]), I, H // 128, *none, *none, 0, p(ws),
                                         ws.numel(), st), "gemm_grouped")
        abi.check(L.qh_silu_mul(p(s["g"]), p(s["u"]), p(s["m"]), M * I, st), "silu_mul")
        abi.check(L.qh_gemm_e4m3_add_rmsnorm(p(s["m"]), p(s["down"][0]), p(s["down"][1]), p(s["o"]), M, H, I, I // 128,
                                             0, p(s["h"]), p(s["norm"]), p(s["hn"]), EPS, p(ws), ws.numel(), st),
                  "gemm_add_rmsnorm")
        return {"h": s["h"], "hn": s["hn"]}
    if k == "attn_decode":
        gate = s["q"].view(-1)[D:]
        abi.check(L.qh_attn_decode(p(s["q"]), 2 * D, p(gate), 2 * D, p(s["k"]), p(s["v"]), p(s["qn"]), p(s["kn"]),
                                   p(s["cos"]), p(s["sin"]), p(s["kc"]), p(s["vc"]), MAX_SEQ, D, ROT, HQ, HKV,
                                   p(s["pos"]), 0, s["splits"], p(s["scratch"]), p(s["counters"]), p(s["out"]), EPS,
                                   st), "attn_decode")
        return {"out": s["out"], "k": s["kc"], "v": s["vc"]}
    if k == "attn":
        M, past = case["M"], case["past"]
        gate = s["q"].view(-1)[D:]
        abi.check(L.qh_attn_prep(p(s["q"]), p(s["k"]), p(s["v"]), p(s["qn"]), p(s["kn"]), p(s["cos"]), p(s["sin"]),
                                 p(s["q32"]), p(s["kc"]), p(s["vc"]), M, HQ, HKV, D, ROT, past, MAX_SEQ, EPS, st),
                  "attn_prep")
        abi.check(L.qh_attn_prefill(p(s["q32"]), p(gate), HQ * 2 * D, 2 * D, p(s["kc"]), p(s["vc"]), p(s["out"]), M,
                                    HQ, HKV, D, past, MAX_SEQ, st), "attn_prefill")
        return {"out": s["out"], "k": s["kc"], "v": s["vc"]}
    # gdn: a new sequence starts from cleared conv and recurrent states
    M = case["M"]
    s["ring"].zero_()
    s["state"].zero_()
    abi.check(L.qh_gdn_prep(p(s["mixed"]), p(s["ring"]), p(s["conv_w"]), p(s["a"]), p(s["b"]), p(s["A_log"]),
                            p(s["dt_bias"]), p(s["y"]), p(s["qn"]), p(s["kn"]), p(s["g"]), p(s["beta"]), M, HK, HV, DL,
                            DL, 0, st), "gdn_prep")
    args = (p(s["qn"]), p(s["kn"]), p(s["y"]), p(s["g"]), p(s["beta"]), p(s["z"]), p(s["norm"]), p(s["state"]),
            p(s["out"]), M, HK, HV, DL, DL, 1e-6)
    if M >= GDN_CHUNK_MIN:
        abi.check(L.qh_gdn_chunk(*args, p(s["ws"]), s["ws"].numel(), st), "gdn_chunk")
    else:
        abi.check(L.qh_gdn_scan(*args, st), "gdn_scan")
    return {"out": s["out"], "state": s["state"], "ring": s["ring"]}


# ---------------------------------------------------------------- what a pass cannot do without

def _layer_linears(i):
    """(N, K) of layer i's projections."""
    mlp = [(I, H), (I, H), (H, I)]
    if CFG.is_full(i):
        return [(CFG.q_proj_rows + 2 * CFG.kv_rows, H), (H, CFG.attn_out_dim)] + mlp
    return [(CONV + CFG.value_dim + 2 * HV, H), (H, CFG.value_dim)] + mlp


def work(case):
    k = case["kind"]
    if k == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        sb = 4 if case["scale"] == "float32" else 2
        ns = math.ceil(N / 128) * (K // 128) if case["mode"] == "block" else N
        return {"bytes": 2 * M * K + N * K + sb * ns + 2 * M * N, "flops": 2 * M * N * K}
    if k in ("mlp", "mlp_decode"):
        M = case.get("M", 1)
        return {"bytes": 3 * I * H * (1 + 4 / 16384) + M * H * 2 * (3 if k == "mlp_decode" else 4) + 4 * H, "flops": 6 * M * I * H}
    if k == "attn_decode":
        c = case["ctx"]
        return {"bytes": 2 * HKV * c * D * 2 + HQ * D * 2 * 3, "flops": 4 * HQ * c * D}
    if k == "attn":
        M, past = case["M"], case["past"]
        pairs = M * past + M * (M + 1) // 2
        return {"bytes": M * HQ * D * 2 * 3 + M * HKV * D * 2 * 4 + past * HKV * D * 4, "flops": 4 * HQ * pairs * D}
    if k == "gdn":
        # per token and head: S^T k, the rank-1 update and S^T q over the 128 x 128 state
        M = case["M"]
        return {"bytes": M * (CONV * 2 + HV * DL * 4 + HV * 4) + HV * DL * DL * 4, "flops": M * HV * 6 * DL * DL}
    wb = sum(n * kk for i in range(CFG.num_hidden_layers) for n, kk in _layer_linears(i))
    M, steps = case["M"], case.get("steps", 0)
    heads = M if k == "score" else 1
    return {"bytes": (1 + steps) * (wb + 2 * V * H) + (heads + steps) * V * 2,
            "flops": 2 * (M + steps) * wb + 2 * (heads + steps) * V * H}


# The relative error of each path against `exact` below (linear 0.0017, MLP 0.0036, attention
# 0.0035, GatedDeltaNet 0.0065: bf16 results and intermediates), about four times over; for whole calls
# the largest that a comparison may allow, since one flipped bf16 rounding in an early layer
# moves every later one.
TOLERANCE = {"linear": 7e-3, "mlp_decode": 1.4e-2, "mlp": 1.4e-2, "attn_decode": 1.4e-2, "attn": 1.4e-2,
             "gdn": 2.4e-2, "chat": 3e-2, "score": 3e-2}


def tolerance(case):
    return {"rel": TOLERANCE[case["kind"]]}


# ---------------------------------------------------------------- the same in 64 bits

def _deq(w, s):
    n, kk = w.shape
    d, s = w.view(torch.float8_e4m3fn).double(), s.double()
    if s.dim() == 1:
        return d * s[:, None]
    return d * s.repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :kk]


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * (1.0 + w.double())


def _rope(x, cos, sin):
    """x [M, heads, D]; cos, sin [M, ROT]: rotate the first ROT dimensions."""
    r, rest = x[..., :ROT], x[..., ROT:]
    half = torch.cat([-r[..., ROT // 2:], r[..., :ROT // 2]], -1)
    return torch.cat([r * cos[:, None].double() + half * sin[:, None].double(), rest], -1)


def _exact_attn(s, M, past):
    q, gate = s["q"].double().split(D, -1)
    at = slice(past, past + M)
    cos, sin = s["cos"][at], s["sin"][at]
    q = _rope(_norm(q, s["qn"]), cos, sin)
    kc, vc = s["kc"].double(), s["vc"].double()
    kc[:, at] = _rope(_norm(s["k"].double(), s["kn"]), cos, sin).transpose(0, 1)
    vc[:, at] = s["v"].double().transpose(0, 1)
    out = torch.empty(M, HQ, D, dtype=torch.float64, device=DEV)
    end = past + M
    mask = torch.arange(end, device=DEV)[None, :] > torch.arange(past, end, device=DEV)[:, None]
    for h in range(HQ):
        kv = h // (HQ // HKV)
        sc = (q[:, h] @ kc[kv, :end].t().contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(sc.masked_fill_(mask, -math.inf), -1) @ vc[kv, :end]
    out = (out * torch.sigmoid(gate)).reshape(M, HQ * D)
    return out, kc, vc


def exact(case, seed):
    k = case["kind"]
    if k in ("chat", "score"):
        return None
    s = _inputs(case, seed)
    if k == "linear":
        return s["x"].double() @ _deq(s["w"], s["s"]).t()
    if k in ("mlp", "mlp_decode"):
        h, x = s["h"].double(), s["x"].double()
        if k == "mlp_decode":
            h = h + x
            x = _norm(h, s["norm"])
        m = torch.nn.functional.silu(x @ _deq(*s["gate"]).t()) * (x @ _deq(*s["up"]).t())
        h = h + m @ _deq(*s["down"]).t()
        return h.view(-1) if k == "mlp_decode" else {"h": h, "hn": _norm(h, s["norm"])}
    if k == "attn_decode":
        out, kc, vc = _exact_attn(s, 1, case["ctx"] - 1)
        return {"out": out.view(-1), "k": kc, "v": vc}
    if k == "attn":
        out, kc, vc = _exact_attn(s, case["M"], case["past"])
        return {"out": out, "k": kc, "v": vc}
    M = case["M"]
    x = torch.cat([torch.zeros(3, CONV, dtype=torch.float64, device=DEV), s["mixed"].double()])
    y = torch.nn.functional.silu(sum(s["conv_w"].double()[:, j] * x[j:j + M] for j in range(4)))
    q, kk, v = y.split([HK * DL, HK * DL, HV * DL], -1)

    def unit(t):
        t = t.view(M, HK, DL)
        t = t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6)
        return t.repeat_interleave(HV // HK, 1)

    q, kk, v = unit(q) / math.sqrt(DL), unit(kk), v.view(M, HV, DL)
    decay = torch.exp(-torch.exp(s["A_log"].double()) * torch.nn.functional.softplus(s["a"].double() + s["dt_bias"].double()))
    beta = torch.sigmoid(s["b"].double())
    S = torch.zeros(HV, DL, DL, dtype=torch.float64, device=DEV)
    o = torch.empty(M, HV, DL, dtype=torch.float64, device=DEV)
    for t in range(M):
        S = S * decay[t, :, None, None]
        d = (v[t] - (S * kk[t, :, :, None]).sum(1)) * beta[t, :, None]
        S = S + kk[t, :, :, None] * d[:, None, :]
        o[t] = (S * q[t, :, :, None]).sum(1)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6) * s["norm"].double()
    out = (o * torch.nn.functional.silu(s["z"].double())).reshape(M, HV * DL)
    ring = torch.zeros(CONV, 4, dtype=torch.float64, device=DEV)
    for t in range(max(0, M - 4), M):
        ring[:, t % 4] = s["mixed"][t].double()
    return {"out": out, "state": S, "ring": ring}
