"""The work a program asks of this framework, as cases that can be prepared, run once and compared.

Kinds (each through the package's public entry points):

  gdn         one token through a run of GDN layers with the mixer's epilogue (`ops.gdn_decode_fused` with z, norm_w),
              recorded once as a HIP graph as a decode loop does; states and conv histories updated in place
  gdn_verify  T tokens through a run of GDN layers, input picked by slot (`ops.gdn_verify_step_slots`), as a graph
  attn        one decode (T = 1) or verify (T > 1) step of a run of attention layers: the mixer with its norms,
              rotation and gate (`ops.attn_mixer_decode`) or the plain call (`ops.paged_gqa_decode`), the new rows
              appended; as a graph, or called directly where "graph" is false
  step        one serving step of a small hybrid stack through the vLLM adapter (`StatePathAdapter.decode_forward`)
  prefill     one GDN layer's prompt (conv, chunked rule) and one attention layer's KV fill, called directly, since
              prompts differ in length
  mlp         the MLP half of a decoder layer over streamed weights (`ops.mlp_decode`)

Sizes are the engine's own: 16 key / 48 value heads of 128, 24 / 4 attention heads of 256, hidden 5120, MLP 17408.
"""
import math
import os
import sys

import torch

_REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_REPO, "tt-qwen-resident_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_REPO, "tt-qwen-resident_amd"))

from qwen36_state import ops  # noqa: E402
from qwen36_state.vllm_adapter import StatePathAdapter  # noqa: E402

NK, NV, D, KC = 16, 48, 128, 4  # key heads, value heads, their dim, conv taps
C = 2 * NK * D + NV * D  # conv channels q | k | v
NQ, NKV, HD, BLK, ROT = 24, 4, 256, 64, 64
EPS = 1e-6
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64


def listed():
    return [
        # every GDN layer of the model for one user: the latency-bound step of interactive use
        dict(name="gdn_b1", kind="gdn", B=1, layers=48),
        # a loaded server: many users, bound by the state's bytes
        dict(name="gdn_b24", kind="gdn", B=24, layers=4),
        # speculative decoding for one user: 3 drafts and a token through 12 GDN layers
        dict(name="gdn_verify_b1_t4", kind="gdn_verify", B=1, T=4, layers=12),
        # a serving step of 8 users of differing context through the adapter (6 GDN + 2 attention layers)
        dict(name="step_b8", kind="step", B=8, ctx=4096, layers=8),
        # a short chat, one attention layer called directly: the smallest call
        dict(name="attn_b1_200", kind="attn", B=1, T=1, ctx=200, ragged=False, mixer=True, pps=8, layers=1, graph=False),
        # one user with a long document
        dict(name="attn_b1_32k", kind="attn", B=1, T=1, ctx=32768, ragged=False, mixer=True, pps=8, layers=2, graph=True),
        # speculative decoding, one user at 8k: 4 rows a step
        dict(name="attn_verify_b1_t4", kind="attn", B=1, T=4, ctx=8192, ragged=False, mixer=True, pps=2, layers=4, graph=True),
        # speculative decoding of a batch with long drafts: 8 rows for each of 4 users of differing context
        dict(name="attn_verify_b4_t8", kind="attn", B=4, T=8, ctx=4100, ragged=True, mixer=False, pps=8, layers=2, graph=True),
        # a chat turn's prompt
        dict(name="prefill_200", kind="prefill", T=200),
        # a long document's prompt
        dict(name="prefill_8192", kind="prefill", T=8192),
        # the MLP half for one user and for a full batch of rows
        dict(name="mlp_b1", kind="mlp", B=1, H=5120, I=17408, gamma=False, down=9),
        dict(name="mlp_b16", kind="mlp", B=16, H=5120, I=17408, gamma=True, down=9),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["gdn", "gdn_verify", "attn", "attn", "step", "prefill", "mlp"])
    if kind == "gdn":
        B = _log_int(rng, 1, 24)
        return dict(kind=kind, B=B, layers=rng.randint(1, max(1, min(48, 96 // B))))
    if kind == "gdn_verify":
        B, T = _log_int(rng, 1, 8), rng.randint(2, 8)
        return dict(kind=kind, B=B, T=T, layers=rng.randint(1, max(1, 48 // (B * T))))
    if kind == "attn":
        B, T = _log_int(rng, 1, 16), rng.choice([1, 1, 1, 2, 3, 4, 5, 6, 8])
        ctx = _log_int(rng, 17, 32768 // B)
        return dict(kind=kind, B=B, T=T, ctx=ctx, ragged=rng.random() < 0.5, mixer=rng.random() < 0.5,
                    pps=rng.choice([2, 4, 8, 8, 16]), layers=rng.randint(1, 4) if B * ctx <= 16384 else 1, graph=True)  # fmt: skip
    if kind == "step":
        return dict(kind=kind, B=_log_int(rng, 1, 8), ctx=_log_int(rng, 100, 4096), layers=rng.choice([4, 8]))
    if kind == "prefill":
        return dict(kind=kind, T=_log_int(rng, 16, 8192))
    return dict(kind=kind, B=_log_int(rng, 1, 16), H=128 * rng.randint(16, 40), I=64 * rng.randint(64, 272),
                gamma=rng.random() < 0.5, down=rng.choice([8, 9]))  # fmt: skip


# ------------------------------------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, *shape, dtype=F32, std=1.0):
    t = torch.empty(shape, dtype=dtype, device="cuda")
    return t.normal_(0.0, std, generator=gen)


def _gates(gen, *shape):
    """Log decay -softplus(n) e^u in (-inf, 0) and beta in (0, 1), as the gate projections give them."""
    u = torch.rand(shape, generator=gen, device="cuda") * -3.0
    g = -torch.nn.functional.softplus(_randn(gen, *shape)) * torch.exp(u)
    return g.contiguous(), torch.sigmoid(_randn(gen, *shape))


def lengths(case):
    """Valid positions of each user after the step's rows: all ctx, or spread evenly over ctx / 4 .. ctx."""
    B, T, ctx = case["B"], case.get("T", 1), case["ctx"]
    if not case.get("ragged", True) or B == 1:
        return [max(T, ctx)] * B
    return [max(T, round(ctx * (0.25 + 0.75 * b / (B - 1)))) for b in range(B)]


def _tables(B, pages, seed, spare=8):
    """Disjoint random pages for every user out of a pool with a few spare ones."""
    nb = B * pages + spare
    perm = torch.randperm(nb, generator=torch.Generator().manual_seed(int(seed)))[: B * pages]
    return perm.view(B, pages).to(torch.int32), nb


def _graph(fn):
    """`fn` recorded once; replayed by every pass."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        with torch.cuda.graph(g, stream=s):
            fn()
    torch.cuda.current_stream().wait_stream(s)
    return g


def _mx_values(w, fmt):
    """fp32 weights [K, N] rounded to values that a microscaling block of 32 along K holds exactly (E2M1, E4M3 or
    two's-complement int8 under one power of two), so the quantized weight equals the weight itself."""
    K, N = w.shape
    b = w.view(K // 32, 32, N)
    emax = {4: 2, 8: 8, 9: 0}[fmt]
    amax = b.abs().amax(1, keepdim=True)
    scale = torch.exp2(torch.floor(torch.log2(amax)) - emax)
    y = b / scale
    if fmt == 4:
        a = y.abs()
        step = torch.where(a < 2, 0.5, torch.where(a < 4, 1.0, 2.0))
        y = torch.sign(y) * (torch.round(a / step) * step).clamp_max(6.0)
    elif fmt == 8:
        y = y.clamp(-448, 448).to(torch.float8_e4m3fn).float()
    else:
        y = torch.round(y * 64).clamp(-127, 127) / 64
    return (y * scale).view(K, N).contiguous()


def _gdn_inputs(case, seed):
    L, B = case["layers"], case["B"]
    gen = _gen(seed)
    s = dict(state=_randn(gen, L, B, NV, D, D, std=0.02), conv=_randn(gen, L, B, C, KC - 1, dtype=BF),
             taps=_randn(gen, L, C, KC, dtype=BF, std=0.5), x=_randn(gen, L, B, C, dtype=BF),
             z=_randn(gen, L, B, NV * D, dtype=BF), norm_w=1 + _randn(gen, L, D, std=0.1))  # fmt: skip
    s["g"], s["beta"] = _gates(gen, L, B, NV)
    return s


def _verify_inputs(case, seed):
    L, B, T = case["layers"], case["B"], case["T"]
    gen = _gen(seed)
    s = dict(states=_randn(gen, L, T, B, NV, D, D, std=0.02), convs=_randn(gen, L, T, B, C, KC - 1, dtype=BF),
             taps=_randn(gen, L, C, KC, dtype=BF, std=0.5), x=_randn(gen, L, B, T, C, dtype=BF))  # fmt: skip
    s["g"], s["beta"] = _gates(gen, L, B, T, NV)
    s["slot"] = torch.randint(0, T, (B,), generator=gen, device="cuda", dtype=torch.int32)
    return s


def _attn_inputs(case, seed):
    L, B, T = case["layers"], case["B"], case["T"]
    gen = _gen(seed)
    lens = lengths(case)
    table, nb = _tables(B, (max(lens) + BLK - 1) // BLK, seed)
    s = dict(kc=_randn(gen, L, nb, NKV, BLK, HD, dtype=BF), vc=_randn(gen, L, nb, NKV, BLK, HD, dtype=BF),
             q=_randn(gen, L, B, T, NQ, HD, dtype=BF), k=_randn(gen, L, B, T, NKV, HD, dtype=BF),
             v=_randn(gen, L, B, T, NKV, HD, dtype=BF), table=table.cuda(),
             lens=torch.tensor(lens, dtype=torch.int32, device="cuda"))  # fmt: skip
    if case["mixer"]:
        s["gate"] = _randn(gen, L, B, T, NQ, HD, dtype=BF)
        s["wq"], s["wk"] = (1 + _randn(gen, L, HD, std=0.1)) / 16, 1 + _randn(gen, L, HD, std=0.1)
        s["pos"] = s["lens"][:, None] - T + torch.arange(T, device="cuda")
    return s


def _prefill_inputs(case, seed):
    T = case["T"]
    gen = _gen(seed)
    table, nb = _tables(1, (T + BLK - 1) // BLK, seed)
    # the projection's output row: q | k | v | z | a | b, of which the conv reads its columns in place
    s = dict(proj=_randn(gen, T, C + NV * D + 2 * NV, dtype=BF), taps=_randn(gen, C, KC, dtype=BF, std=0.5),
             k=_randn(gen, NKV, T, HD, dtype=BF), v=_randn(gen, NKV, T, HD, dtype=BF), table=table[0].cuda().contiguous(),
             kc=torch.zeros(nb, NKV, BLK, HD, dtype=BF, device="cuda"),
             vc=torch.zeros(nb, NKV, BLK, HD, dtype=BF, device="cuda"))  # fmt: skip
    s["g"], s["beta"] = _gates(gen, T, NV)
    return s


def _mlp_inputs(case, seed):
    B, H, I = case["B"], case["H"], case["I"]
    gen = _gen(seed)
    s = dict(x=_randn(gen, B, H), gamma=1 + _randn(gen, H, std=0.1) if case["gamma"] else None)
    for name, (k, n), fmt, std in (("gate", (H, I), 4, H**-0.5), ("up", (H, I), 4, H**-0.5),
                                   ("down", (I, H), case["down"], I**-0.5)):  # fmt: skip
        s[name] = _mx_values(_randn(gen, k, n, std=std), fmt)
    return s


def _step_inputs(case, seed):
    """Per layer the resident tensors and this step's inputs, in layer order."""
    B, L = case["B"], case["layers"]
    gen = _gen(seed)
    lens = lengths(case)
    table, nb = _tables(B, (case["ctx"] + BLK - 1) // BLK, seed)
    lay = []
    for l in range(L):
        if (l + 1) % 4 == 0:
            lay.append(dict(attn=True, kc=_randn(gen, nb, NKV, BLK, HD, dtype=BF), vc=_randn(gen, nb, NKV, BLK, HD, dtype=BF),
                            q=_randn(gen, B, 1, NQ, HD, dtype=BF), k_new=_randn(gen, B, 1, NKV, HD, dtype=BF),
                            v_new=_randn(gen, B, 1, NKV, HD, dtype=BF)))  # fmt: skip
        else:
            d = dict(attn=False, state=_randn(gen, B, NV, D, D, std=0.02), conv=_randn(gen, B, C, KC - 1, dtype=BF),
                     taps=_randn(gen, C, KC, dtype=BF, std=0.5), x=_randn(gen, B, C, dtype=BF))  # fmt: skip
            d["g"], d["beta"] = _gates(gen, B, NV)
            lay.append(d)
    return dict(layers=lay, table=table, nb=nb, lens=lens)


# ------------------------------------------------------------------------------------------- prepare and run


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gdn":
        s = _gdn_inputs(case, seed)
        L, B = case["layers"], case["B"]
        s["o"] = torch.empty(L, B, NV, D, dtype=BF, device="cuda")
        s["ws"] = torch.zeros(max(256, ops.lib().qs_gdn_workspace_bytes(B, NK)), dtype=torch.uint8, device="cuda")

        def layers():
            for l in range(L):
                ops.gdn_decode_fused(s["x"][l], s["conv"][l], s["taps"][l], s["g"][l], s["beta"][l], s["state"][l],
                                     out=s["o"][l], ws=s["ws"], z=s["z"][l], norm_w=s["norm_w"][l])  # fmt: skip

        s["graph"] = _graph(layers)
    elif kind == "gdn_verify":
        s = _verify_inputs(case, seed)
        L, B, T = case["layers"], case["B"], case["T"]
        s["out"] = (torch.empty(L, B, T, NV, D, dtype=BF, device="cuda"), torch.empty_like(s["states"]),
                    torch.empty_like(s["convs"]))  # fmt: skip

        def layers():
            for l in range(L):
                ops.gdn_verify_step_slots(s["x"][l], s["convs"][l], s["taps"][l], s["g"][l], s["beta"][l], s["states"][l],
                                          s["slot"], out=tuple(t[l] for t in s["out"]))  # fmt: skip

        s["graph"] = _graph(layers)
    elif kind == "attn":
        s = _attn_inputs(case, seed)
        B, T, pps = case["B"], case["T"], case["pps"]
        s["o"] = torch.empty_like(s["q"])
        nbytes = ops.lib().qs_paged_attention_workspace_bytes(B, T, NQ, NKV, HD, s["table"].shape[1], pps)
        s["ws"] = torch.zeros(max(256, nbytes), dtype=torch.uint8, device="cuda")
        if case["mixer"]:
            s["cos"], s["sin"] = ops.rope_tables(s["pos"])

        def layers():
            for l in range(case["layers"]):
                if case["mixer"]:
                    ops.attn_mixer_decode(s["q"][l], s["k"][l], s["v"][l], s["gate"][l], s["wq"][l], s["wk"][l], s["cos"],
                                          s["sin"], s["kc"][l], s["vc"][l], s["table"], s["lens"], pages_per_split=pps,
                                          out=s["o"][l], ws=s["ws"])  # fmt: skip
                else:
                    ops.paged_gqa_decode(s["q"][l], s["kc"][l], s["vc"][l], s["table"], s["lens"], HD**-0.5, k_new=s["k"][l],
                                         v_new=s["v"][l], pages_per_split=pps, out=s["o"][l], ws=s["ws"])  # fmt: skip

        # the state never holds both the graph and the closure over it: a cycle would leave the graph to the garbage
        # collector, which may destroy it while another one is being recorded, an error that ends the process
        if case["graph"]:
            s["graph"] = _graph(layers)
        else:
            s["call"] = layers
    elif kind == "step":
        d = _step_inputs(case, seed)
        gdn = [x for x in d["layers"] if not x["attn"]]
        att = [x for x in d["layers"] if x["attn"]]
        ad = StatePathAdapter(case["B"], d["table"].shape[1] * BLK, layers=case["layers"], device="cuda:0",
                              taps=[x["taps"] for x in gdn])  # fmt: skip
        kv = ad.allocate_kv_cache((d["nb"], NKV, BLK, HD), BF, len(att))
        for (kc, vc), x in zip(kv, att):
            kc.copy_(x["kc"])
            vc.copy_(x["vc"])
        for i, x in enumerate(gdn):
            ad.gdn_state[i].copy_(x["state"])
            ad.conv_state[i].copy_(x["conv"])
        ad.block_table.copy_(d["table"])
        for buf, x in zip(ad.step_inputs(), d["layers"]):
            for key, t in buf.items():
                t.copy_(x[key])
        s = dict(ad=ad, kv=kv, pos=torch.tensor(d["lens"], dtype=torch.int32) - 1)
    elif kind == "prefill":
        s = _prefill_inputs(case, seed)
        s["x"] = s["proj"][:, :C]
        s["conv"] = torch.empty(C, KC - 1, dtype=BF, device="cuda")
        s["state"] = torch.empty(NV, D, D, device="cuda")
    else:
        s = _mlp_inputs(case, seed)
        for name, fmt in (("gate", 4), ("up", 4), ("down", case["down"])):
            s[name] = ops.MxWeight.quantize(s[name], fmt)
        s["out"] = torch.empty_like(s["x"])
    s["kind"] = kind
    return s


def run(s):
    kind = s["kind"]
    if kind == "gdn":
        s["graph"].replay()
        return dict(o=s["o"], state=s["state"], conv=s["conv"])
    if kind == "gdn_verify":
        s["graph"].replay()
        return dict(o=s["out"][0], states=s["out"][1], convs=s["out"][2])
    if kind == "attn":
        if "graph" in s:
            s["graph"].replay()
        else:
            s["call"]()
        return dict(o=s["o"], kc=s["kc"], vc=s["vc"])
    if kind == "step":
        outs = s["ad"].decode_forward(None, s["pos"])
        return dict(o=outs, state=s["ad"].gdn_state, conv=s["ad"].conv_state, kv=s["kv"])
    if kind == "prefill":
        q, k, v, _ = ops.causal_conv1d_prefill(s["x"], s["taps"], None, s["conv"])
        o, state = ops.chunk_gated_delta_rule(q, k, v, s["g"], s["beta"], final_state=s["state"])
        ops.paged_kv_fill(s["k"], s["v"], s["kc"], s["vc"], s["table"])
        return dict(o=o, state=state, conv=s["conv"], kc=s["kc"], vc=s["vc"])
    return dict(out=ops.mlp_decode(s["x"], s["gamma"], s["gate"], s["up"], s["down"], out=s["out"]))


# ------------------------------------------------------------------------------------- work and tolerances


def _gdn_work(B, T, writes, epilogue):
    """Bytes of one GDN layer: state and conv history read once and written `writes` times, taps, x, gates, o (and
    with the epilogue z and its norm weight); two flops for each of k^T S, the decay, the update and q^T S."""
    state, conv = B * NV * D * D * 4, B * C * (KC - 1) * 2
    nbytes = (1 + writes) * (state + conv) + C * KC * 2 + B * T * (C * 2 + NV * 8 + NV * D * 2)
    if epilogue:
        nbytes += B * NV * D * 2 + D * 4
    return nbytes, B * T * NV * 7 * D * D


def _attn_work(case, mixer):
    """K and V of every valid position, the new rows read and stored, q, o (and the gate), the table."""
    B, T, row = case["B"], case.get("T", 1), NKV * HD * 2
    lens = lengths(case)
    nbytes = sum(2 * n * row + (n + BLK - 1) // BLK * 4 for n in lens)
    nbytes += B * T * (4 * row + (3 if mixer else 2) * NQ * HD * 2)
    return nbytes, 4 * T * NQ * HD * sum(lens)


def work(case):
    kind = case["kind"]
    if kind == "gdn":
        n, f = _gdn_work(case["B"], 1, 1, True)
        n, f = n * case["layers"], f * case["layers"]
    elif kind == "gdn_verify":
        n, f = _gdn_work(case["B"], case["T"], case["T"], False)
        n, f = n * case["layers"], f * case["layers"]
    elif kind == "attn":
        n, f = _attn_work(case, case["mixer"])
        n, f = n * case["layers"], f * case["layers"]
    elif kind == "step":
        na = case["layers"] // 4
        gn, gf = _gdn_work(case["B"], 1, 1, False)
        an, af = _attn_work(case, False)
        n, f = na * an + (case["layers"] - na) * gn, na * af + (case["layers"] - na) * gf
    elif kind == "prefill":
        T = case["T"]
        n = T * (C * 2 + NV * 8 + NV * D * 2) + C * KC * 2 + C * (KC - 1) * 2 + NV * D * D * 4 + 2 * 2 * T * NKV * HD * 2
        f = T * NV * 6 * D * D
    else:
        B, H, I = case["B"], case["H"], case["I"]
        n = 2 * (H * I // 2 + H * I // 32) + I * H + I * H // 32 + 2 * B * H * 4 + (H * 4 if case["gamma"] else 0)
        f = 6 * B * H * I
    return dict(bytes=n, flops=f)


def tolerance(case):
    """Four times what each kind measured against 64 bits: one rounding to bf16 of the GDN and prefill outputs
    (1.7e-3; the fp32 states beside them 3e-6 .. 9e-5), attention's bf16 probabilities on top of that (2.3e-3), the
    MLP's bf16 h and z (1.5e-3)."""
    return {"rel": {"attn": 1e-2, "step": 1e-2, "mlp": 6e-3}.get(case["kind"], 7e-3)}


# ------------------------------------------------------------------------------------------- 64-bit results


def _bf(t):
    return t.to(F32).to(BF).to(F64)


def _silu(t):
    return t * torch.sigmoid(t)


def _rms(t, w):
    return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + EPS) * w


def _conv(window, taps):
    """window [..., C, 4 inputs], oldest first -> silu(sum), rounded to bf16 as the path hands it on."""
    return _bf(_silu((window * taps).sum(-1)))


def _rule(y, g, beta, S):
    """One token of the gated delta rule: y [..., C], S [..., NV, D, D] -> o, S'."""
    q, k, v = y[..., : NK * D], y[..., NK * D : 2 * NK * D], y[..., 2 * NK * D :]
    unit = lambda t: t * torch.rsqrt(t.square().sum(-1, keepdim=True) + EPS)  # noqa: E731
    q = unit(q.unflatten(-1, (NK, D))).repeat_interleave(NV // NK, -2) * D**-0.5
    k = unit(k.unflatten(-1, (NK, D))).repeat_interleave(NV // NK, -2)
    v = v.unflatten(-1, (NV, D))
    S = S * g.exp()[..., None, None]
    delta = beta[..., None] * (v - (k[..., None] * S).sum(-2))
    S = S + k[..., None] * delta[..., None, :]
    return (q[..., None] * S).sum(-2), S


def _gdn_exact(x, conv, taps, g, beta, S):
    window = torch.cat([conv.double(), x.double()[..., None]], -1)
    o, S = _rule(_conv(window, taps.double()), g.double(), beta.double(), S.double())
    return o, S, window[..., 1:]


def _rope(t, pos):
    """The first ROT dims of each head rotated, halves paired; pos [B, T]."""
    inv = 1.0 / ops.ROPE_THETA ** (torch.arange(0, ROT, 2, dtype=F64, device=t.device) / ROT)
    ang = (pos.double()[..., None] * inv)[:, :, None]
    a, b = t[..., : ROT // 2], t[..., ROT // 2 : ROT]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin(), t[..., ROT:]], -1)


def _append(pool, rows, table, lens):
    """`rows` [B, T, NKV, HD] at positions lens - T .. lens - 1 of each user's pages."""
    T = rows.shape[1]
    for b, n in enumerate(lens):
        for t in range(T):
            p = n - T + t
            pool[int(table[b, p // BLK]), :, p % BLK] = rows[b, t]
    return pool


def _attend(q, kc, vc, table, lens):
    """softmax(q K^T) V of one layer over each user's pages, causal among its new rows; q [B, T, NQ, HD] scaled."""
    B, T = q.shape[:2]
    out = torch.empty_like(q)
    for b, n in enumerate(lens):
        rows = table[b, : (n + BLK - 1) // BLK].long()
        K = kc[rows].permute(1, 0, 2, 3).reshape(NKV, -1, HD)[:, :n].double()
        V = vc[rows].permute(1, 0, 2, 3).reshape(NKV, -1, HD)[:, :n].double()
        qq = q[b].view(T, NKV, NQ // NKV, HD).permute(1, 0, 2, 3).reshape(NKV, -1, HD).contiguous()
        s = (qq @ K.transpose(1, 2).contiguous()).view(NKV, T, NQ // NKV, n)
        seen = torch.arange(n, device=q.device) <= (n - T + torch.arange(T, device=q.device))[:, None]
        p = s.masked_fill(~seen[None, :, None], -math.inf).softmax(-1).view(NKV, -1, n)
        out[b] = (p @ V).view(NKV, T, NQ // NKV, HD).permute(1, 0, 2, 3).reshape(T, NQ, HD)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "gdn":
        s = _gdn_inputs(case, seed)
        o, S, conv = [], [], []
        for l in range(case["layers"]):
            a, b, c = _gdn_exact(s["x"][l], s["conv"][l], s["taps"][l], s["g"][l], s["beta"][l], s["state"][l])
            o.append(_rms(a, s["norm_w"][l].double()) * _silu(s["z"][l].double().view_as(a)))
            S.append(b)
            conv.append(c)
        return dict(o=torch.stack(o), state=torch.stack(S), conv=torch.stack(conv))
    if kind == "gdn_verify":
        s = _verify_inputs(case, seed)
        B, T = case["B"], case["T"]
        o, S, conv = [], [], []
        for l in range(case["layers"]):
            pick = s["slot"].long(), torch.arange(B, device="cuda")
            st, cv, ol, sl, cl = s["states"][l][pick], s["convs"][l][pick], [], [], []
            for t in range(T):
                a, st, cv = _gdn_exact(s["x"][l, :, t], cv, s["taps"][l], s["g"][l, :, t], s["beta"][l, :, t], st)
                ol.append(a)
                sl.append(st)
                cl.append(cv)
            o.append(torch.stack(ol, 1))
            S.append(torch.stack(sl))
            conv.append(torch.stack(cl))
        return dict(o=torch.stack(o), states=torch.stack(S), convs=torch.stack(conv))
    if kind == "attn":
        s = _attn_inputs(case, seed)
        lens, o, ks, vs = lengths(case), [], [], []
        for l in range(case["layers"]):
            q, k = s["q"][l].double() * HD**-0.5, s["k"][l].double()
            if case["mixer"]:
                q = _rope(_rms(s["q"][l].double(), s["wq"][l].double()), s["pos"])
                k = _bf(_rope(_rms(k, s["wk"][l].double()), s["pos"]))
            kc = _append(s["kc"][l], k.to(BF), s["table"], lens)
            vc = _append(s["vc"][l], s["v"][l], s["table"], lens)
            a = _attend(q, kc, vc, s["table"], lens)
            o.append(a * torch.sigmoid(s["gate"][l].double()) if case["mixer"] else a)
        return dict(o=torch.stack(o), kc=s["kc"].double(), vc=s["vc"].double())
    if kind == "step":
        d = _step_inputs(case, seed)
        o, S, conv, kv = [], [], [], []
        for x in d["layers"]:
            if x["attn"]:
                kc = _append(x["kc"], x["k_new"], d["table"], d["lens"])
                vc = _append(x["vc"], x["v_new"], d["table"], d["lens"])
                o.append(_attend(x["q"].double() * HD**-0.5, kc, vc, d["table"].cuda(), d["lens"]))
                kv.append((kc.double(), vc.double()))
            else:
                a, b, c = _gdn_exact(x["x"], x["conv"], x["taps"], x["g"], x["beta"], x["state"])
                o.append(a)
                S.append(b)
                conv.append(c)
        return dict(o=o, state=torch.stack(S), conv=torch.stack(conv), kv=kv)
    if kind == "prefill":
        s = _prefill_inputs(case, seed)
        T = case["T"]
        x = torch.cat([torch.zeros(KC - 1, C, dtype=F64, device="cuda"), s["proj"][:, :C].double()])
        y = torch.empty(T, C, dtype=F64, device="cuda")
        for t0 in range(0, T, 1024):
            n = min(1024, T - t0)
            y[t0 : t0 + n] = _conv(x[t0 : t0 + n + KC - 1].unfold(0, KC, 1), s["taps"].double())
        S, o = torch.zeros(NV, D, D, dtype=F64, device="cuda"), torch.empty(T, NV, D, dtype=F64, device="cuda")
        g, beta = s["g"].double(), s["beta"].double()
        for t in range(T):
            o[t], S = _rule(y[t], g[t], beta[t], S)
        pools = []
        for rows, pool in ((s["k"], s["kc"]), (s["v"], s["vc"])):
            pos = torch.arange(T, device="cuda")
            pool[s["table"][pos // BLK].long(), :, pos % BLK] = rows.transpose(0, 1)
            pools.append(pool.double())
        return dict(o=o, state=S, conv=x[T:].t().contiguous(), kc=pools[0], vc=pools[1])
    s = _mlp_inputs(case, seed)
    x = s["x"].double()
    h = _rms(x, s["gamma"].double() if case["gamma"] else 1.0)
    z = _silu(h @ s["gate"].double()) * (h @ s["up"].double())
    return dict(out=x + z @ s["down"].double())
