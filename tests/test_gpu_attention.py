"""Paged GQA decode attention on the GPU against the oracle (gather + fp32 softmax over the pages):
bf16 output rtol 2e-2; the fused append leaves the pools bit-identical to the oracle's append."""
import pytest
import torch
from conftest import assert_attn_output

from oracle import state_path as O
from qwen36_state import ops, workloads as W

pytestmark = pytest.mark.gpu

CNT_BYTES = 65536  # the fixed counter block at the head of an attention workspace


def pairs(T, G, mixer):
    """Whether a verify step (more than 16 query rows per KV head) can walk two pages at once."""
    R = T * G
    nrb = -(-R // 64)
    tiles = -(-R // (16 * nrb))
    return not mixer or tiles == 2 or (tiles == 3 and T <= 8)


def plan(B, T, G, width, pps, mixer=False, nkv=4):
    """How a call with a workspace is cut (the rules of the library's launch): pages a workgroup walks, splits, and
    whether the attention launch merges them itself. The tests below choose their shapes by it."""
    R = T * G
    few = B * nkv <= 16
    whole = (3 if few and not mixer else 2) if R <= 8 else (4 if few else 3) if R <= 16 else 2 if pairs(T, G, mixer) else 1
    if width <= min(whole, pps):
        return width, 1, False
    most = 256 // (B * nkv * -(-R // 64))
    p = -(-width // most) if most else pps
    p = min(pps, p if p <= 1 or not most else p + p % 2)
    ns = -(-width // p)
    wpp = 2 if p > 1 else 1
    rows, wgs = -(-R // (4 * wpp)), B * nkv * ns
    few = wgs * rows * rows <= 192 or rows == 1 and (T > 2 or wpp == 1 and wgs > 256)
    return p, ns, 1 < ns and R <= 16 and (ns <= 4 or R <= 8 * wpp and (ns <= 8 or ns <= 16 and few))


def split_rows(ws):
    """The rows of split partials a call wrote (every split holding pages) into a workspace whose bytes past the counters
    were 0xFF, from the first float that is still a NaN: 2 floats (m, l) a row, padded to 256 bytes, then 256 of O."""
    nan = ws[CNT_BYTES:].view(torch.float32).isnan().cpu()
    n = int(nan.float().argmax()) if bool(nan.any()) else len(nan)
    return n // 2 if n % 64 else n // 258


def run_case(dev, d, pps, fused=True):
    """Attention (+ append) on the GPU and the same step through the oracle; returns (o_gpu, o_ref,
    pools equal)."""
    g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
    B, T = d["q"].shape[:2]
    pos = d["seq_lens"] - T
    if fused:
        o = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"],
                                 k_new=g["k_new"], v_new=g["v_new"], pages_per_split=pps)  # fmt: skip
    else:
        ops.paged_kv_append(g["k_new"], g["v_new"], g["k_cache"], g["v_cache"], g["block_table"], pos.to(dev))
        o = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"],
                                 pages_per_split=pps)  # fmt: skip
    kc, vc = d["k_cache"].clone(), d["v_cache"].clone()
    O.paged_append(kc, vc, d["k_new"], d["v_new"], d["block_table"], pos)
    o_ref = O.gqa_decode(d["q"], kc, vc, d["block_table"], d["seq_lens"], d["scale"])
    same = torch.equal(g["k_cache"].cpu(), kc) and torch.equal(g["v_cache"].cpu(), vc)
    return o, O.bf16(o_ref), same


@pytest.mark.parametrize(
    "B,ctx,T,pps",
    [
        (1, 32768, 1, 8),  # the 32k layer as benchmarked: 512 pages, 64 splits through the merge launch
        (8, 4096, 1, 8),  # the batch-8 step's layer as benchmarked: 8 splits merged inside the launch
        (8, 4096, 1, 4),  # 16 splits, merged in a launch of their own
        (1, 8192, 4, 8),  # verify: 4 new rows, causal among them (24 query rows per KV head)
        (1, 32768, 1, 1),  # 512 splits (2048 workgroups) through the merge launch
        (2, 4096, 1, 64),  # one split: no merge
        (2, 3000, 6, 4),  # 36 query rows per KV head: three tiles of the rows kernel
        (1, 700, 7, 64),  # three tiles, odd token count, one split
        (3, 900, 2, 4),  # 12 query rows per KV head: two tokens on the one-token kernel
        (2, 60, 1, 8),  # a one-page table without a workspace: one page per workgroup, one token
        (2, 60, 3, 8),  # and three
    ],
)
def test_attention(dev, B, ctx, T, pps):
    d = W.attn_layer(B, ctx, "cpu", seed=B + ctx + T + pps, T=T)
    o, o_ref, same = run_case(dev, d, pps)
    assert same
    assert_attn_output(o, o_ref)


def test_attention_ragged_users(dev):
    """Users at different lengths (1 position, exactly one page, one past a page, mid-page) in one launch."""
    d = W.attn_layer(4, 11 * 64, "cpu", seed=77, T=1, num_blocks=64)
    d["seq_lens"] = torch.tensor([1, 64, 65, 700], dtype=torch.int32)
    o, o_ref, same = run_case(dev, d, pps=2)
    assert same
    assert_attn_output(o, o_ref)
    # a user with a single position attends only to its new row: o = v_new exactly (up to bf16 rounding)
    torch.testing.assert_close(o[0, 0].cpu().float(), d["v_new"][0, 0].float().repeat_interleave(6, 0), rtol=0, atol=0)


# The pages a workgroup walks follow the grid: 8 users of 8 pages at 2 pages per split are cut to one page (256
# workgroups), 9 users keep two (288 would be past them); 64 users keep one split of 5 pages each, 70 users two splits of
# up to 4 pages, walked two at a time, at 1, 4 and 8 tokens (6, 24 and 48 query rows per KV head); 4 users of 65 pages
# walk 6 of the caller's 8, 5 users of 50 the caller's 5
@pytest.mark.parametrize("B,pages,T,pps", [(8, 8, 1, 2), (9, 8, 1, 2), (64, 5, 1, 8), (70, 5, 1, 4), (70, 5, 4, 4),
                                           (70, 5, 8, 4), (1, 20, 1, 7), (2, 30, 5, 16), (4, 65, 8, 8),
                                           (5, 50, 1, 5)])  # fmt: skip
def test_attention_walked_pages(dev, B, pages, T, pps):
    d = W.attn_layer(B, pages * 64, "cpu", seed=B + T, T=T, num_blocks=B * pages + 8)
    gen = torch.Generator().manual_seed(B)
    d["seq_lens"] = torch.randint(T, pages * 64 + 1, (B,), generator=gen).to(torch.int32)
    o, o_ref, same = run_case(dev, d, pps)
    assert same
    assert_attn_output(o, o_ref)


def test_attention_unfused_equals_fused(dev):
    d = W.attn_layer(2, 1000, "cpu", seed=5, T=2, num_blocks=64)
    o1, ref, _ = run_case(dev, d, pps=4, fused=True)
    o2, _, same = run_case(dev, d, pps=4, fused=False)
    assert same
    assert torch.equal(o1.cpu(), o2.cpu())
    assert_attn_output(o1, ref)


@pytest.mark.parametrize(
    "G,T,lens,pps",
    [
        (6, 4, [8194], 2),  # the verify shape; new rows at 62..65 of a page pair
        (6, 4, [8194], 1),  # each of those pages its own split
        (6, 5, [700, 337, 4099], 4),  # ragged users: new rows inside one slice, across slices, across pages
        (6, 3, [337], 64),  # one split (no merge); rows 14..16 span two waves' slices
        (4, 8, [1000, 9 * 64 + 4], 2),  # 8 new rows, the most of the form for few; the second user's span pages
        (8, 4, [130, 64], 1),  # 32 query rows; the second user's new rows end its only page
        (2, 9, [777], 2),  # 9 new rows: the form for up to 16
        (2, 16, [2000], 4),  # the most new rows a call takes (16)
    ],
)
def test_verify_append_from_registers(dev, G, T, lens, pps):
    """The rows kernel (here 17 to 32 query rows per KV head) attends the step's new rows from LDS (the new K rows
    over the score operand's, the new V rows as the page is staged) and writes them to the pool after the page loop:
    output bit-equal to the unfused append followed by attention, pools equal to the oracle's append, output within
    the oracle's tolerance."""
    d = W.attn_layer(len(lens), max(lens), "cpu", seed=G * 100 + T + pps, T=T, num_blocks=512)
    d["seq_lens"] = torch.tensor(lens, dtype=torch.int32)
    nkv = d["k_cache"].shape[1]
    q = d["q"] if G * nkv <= d["q"].shape[2] else torch.cat([d["q"], d["q"]], dim=2)
    d["q"] = q[:, :, : G * nkv].contiguous()
    assert 16 < T * G <= 32
    o1, ref, same1 = run_case(dev, d, pps, fused=True)
    o2, _, same2 = run_case(dev, d, pps, fused=False)
    assert same1 and same2
    assert torch.equal(o1.cpu(), o2.cpu())
    assert_attn_output(o1, ref)


def test_attention_repeatable(dev):
    d = W.attn_layer(1, 32768, "cpu", seed=9)
    g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
    outs = [
        ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"],
                             k_new=g["k_new"], v_new=g["v_new"], pages_per_split=8).cpu()  # fmt: skip
        for _ in range(3)
    ]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[1], outs[2])


@pytest.mark.parametrize("B,ctx,T,pps", [(2, 1000, 1, 4), (1, 2048, 3, 2), (3, 700, 2, 64), (1, 900, 6, 4)])
def test_attn_mixer(dev, B, ctx, T, pps):
    """q/k RMSNorm + partial RoPE and the sigmoid gate around the paged attention (model.py:237-246), one and two
    tokens, three and six (18 and 36 rows, the rows kernel), each a page per split: the appended K rows within
    one bf16 ulp of the oracle's (rsqrt and the rotation differ in the last fp32 bits between libraries), V
    rows bit-exact, the output rtol 2e-2."""
    from conftest import bf16_ulp_mismatch

    d = W.attn_layer(B, ctx, "cpu", seed=ctx + T, T=T, num_blocks=64)
    gen = torch.Generator().manual_seed(ctx)
    gate = torch.randn(d["q"].shape, generator=gen).bfloat16()
    wq = (1 + 0.1 * torch.randn(256, generator=gen)) / 16.0
    wk = 1 + 0.1 * torch.randn(256, generator=gen)
    pos = (d["seq_lens"] - T)[:, None] + torch.arange(T)[None]
    cos, sin = O.rope_tables(pos + 5000)
    g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
    o = ops.attn_mixer_decode(g["q"], g["k_new"], g["v_new"], gate.to(dev), wq.to(dev), wk.to(dev), cos.to(dev),
                              sin.to(dev), g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"],
                              pages_per_split=pps)  # fmt: skip
    kc, vc = d["k_cache"].clone(), d["v_cache"].clone()
    o_ref = O.attn_mixer(d["q"], d["k_new"], d["v_new"], gate, wq, wk, cos, sin, kc, vc, d["block_table"],
                         d["seq_lens"])  # fmt: skip
    assert torch.equal(g["v_cache"].cpu(), vc)
    ulps, frac = bf16_ulp_mismatch(g["k_cache"].cpu(), kc)
    assert ulps <= 1 and frac < 1e-3, (ulps, frac)
    assert_attn_output(o, o_ref)
    # the rope tables of the wrapper equal the oracle's
    c2, s2 = ops.rope_tables(pos.to(dev) + 5000)
    assert torch.equal(c2.cpu(), cos) and torch.equal(s2.cpu(), sin)


def test_in_launch_merge_counters_rearm(dev):
    """Few splits are merged inside the attention launch by the last workgroup to arrive. The arrival counters at the
    workspace head read zero after every call, so one workspace serves repeated calls and calls of other shapes (here
    8, 5 and 4 splits of batch 8, 3 and 6, one and two tokens, twice each): outputs repeat bit-exactly and match the
    oracle."""
    L = ops.lib()
    cases = [(8, 4096, 1, 8, 8), (3, 300, 1, 4, 5), (6, 250, 2, 2, 4)]  # users, positions, tokens, pages, splits
    assert all(plan(B, T, 6, -(-ctx // 64), pps)[1:] == (ns, True) for B, ctx, T, pps, ns in cases)
    nbytes = max(L.qs_paged_attention_workspace_bytes(B, T, 24, 4, 256, -(-ctx // 64), pps) for B, ctx, T, pps, _ in cases)
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    data = [W.attn_layer(B, ctx, "cpu", seed=B + T, T=T, num_blocks=1024) for B, ctx, T, _, _ in cases]
    outs = []
    for rep in range(2):
        for d, (_, _, _, pps, _) in zip(data, cases):
            g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
            o = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"],
                                     pages_per_split=pps, ws=ws)  # fmt: skip
            torch.cuda.synchronize()
            assert int(ws[:CNT_BYTES].view(torch.int32).abs().sum()) == 0, "counters not re-armed"
            outs.append(o.cpu())
    n = len(cases)
    assert all(torch.equal(outs[i], outs[i + n]) for i in range(n))
    for d, o in zip(data, outs):
        ref = O.gqa_decode(d["q"], d["k_cache"], d["v_cache"], d["block_table"], d["seq_lens"], d["scale"])
        assert_attn_output(o, O.bf16(ref))


# Where the merge moves between the launches: 4 and 5 splits of 12 rows and 8 and 9 of 6 on one page per workgroup (9 at
# batch 1 in the launch), 8 and 9 of 12 rows on two pages, 2 splits of 16 rows (group size 8) and of 18; 16 splits in the
# launch for 4 rows at batch 1, one row at batch 3 and, past a workgroup per CU, 5, but not 4, and 4 tokens of one head, or
# 8 of them on two pages, at batch 4, not for 8 rows. And where a table stays whole: 2 and 3 pages of 6 rows at batch 4, 2
# but not 3 at batch 5, 4 but not 5 of 12 rows at batch 4, 3 but not 4 at batch 5, 2 but not 3 of 24. The partials written
# show the split count.
@pytest.mark.parametrize("B,G,T,width,pps,splits,merged", [
    (6, 6, 2, 4, 2, 4, True), (2, 6, 2, 5, 2, 5, False), (2, 6, 1, 8, 8, 8, True), (2, 6, 1, 9, 8, 9, False),
    (1, 6, 1, 9, 8, 9, True), (1, 4, 1, 16, 8, 16, True), (3, 1, 1, 16, 1, 16, True), (4, 1, 1, 16, 8, 16, False),
    (5, 1, 1, 16, 1, 16, True), (1, 8, 1, 16, 8, 16, False), (4, 1, 4, 16, 8, 16, True), (4, 1, 8, 64, 8, 16, True),
    (8, 6, 2, 16, 2, 8, True), (7, 6, 2, 18, 8, 9, False), (64, 8, 2, 5, 4, 2, True), (64, 6, 3, 5, 4, 2, False),
    (4, 6, 1, 1, 8, 1, False), (4, 6, 1, 2, 2, 1, False), (4, 6, 1, 3, 8, 1, False), (4, 6, 1, 3, 2, 3, True),
    (5, 6, 1, 2, 8, 1, False), (5, 6, 1, 3, 8, 3, True), (4, 6, 2, 4, 8, 1, False), (4, 6, 2, 5, 8, 5, False),
    (5, 6, 2, 3, 8, 1, False), (5, 6, 2, 4, 8, 4, True), (1, 6, 4, 2, 8, 1, False), (1, 6, 4, 3, 8, 3, False),
    (1, 6, 8, 2, 8, 1, False), (1, 6, 11, 2, 8, 1, False), (1, 6, 11, 3, 8, 3, False),
])  # fmt: skip
@pytest.mark.parametrize("mixer", [False, True])
def test_split_plans(dev, B, G, T, width, pps, splits, merged, mixer):
    if mixer and (B, T, width, pps) == (4, 1, 3, 8):
        splits, merged = 3, True  # the mixer's launch keeps 2 pages whole, not 3
    if mixer and (T, width) == (11, 2):
        splits = 2  # and of 11 tokens, whose rows it walks a page at a time, none
    assert plan(B, T, G, width, pps, mixer)[1:] == (splits, merged)
    d = W.attn_layer(B, width * 64, "cpu", seed=B + T + width, T=T, num_blocks=B * width + 8)
    gen = torch.Generator().manual_seed(width)
    d["q"] = torch.randn(B, T, G * 4, 256, generator=gen).bfloat16()
    d["seq_lens"] = torch.randint((width - 1) * 64 + T, width * 64 + 1, (B,), generator=gen).to(torch.int32)
    ws = torch.zeros(ops.lib().qs_paged_attention_workspace_bytes(B, T, G * 4, 4, 256, width, pps), dtype=torch.uint8,
                     device=dev)  # fmt: skip
    ws[CNT_BYTES:] = 0xFF
    if mixer:
        check_mixer(dev, d, pps, 64, gen, ws=ws)
    else:
        g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
        o = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"],
                                 k_new=g["k_new"], v_new=g["v_new"], pages_per_split=pps, ws=ws)  # fmt: skip
        kc, vc = d["k_cache"].clone(), d["v_cache"].clone()
        O.paged_append(kc, vc, d["k_new"], d["v_new"], d["block_table"], d["seq_lens"] - T)
        assert_attn_output(o, O.bf16(O.gqa_decode(d["q"], kc, vc, d["block_table"], d["seq_lens"], d["scale"])))
    assert split_rows(ws) == (B * 4 * splits * T * G if splits > 1 else 0)
    assert int(ws[:CNT_BYTES].view(torch.int32).abs().sum()) == 0, "counters not re-armed"


# More splits go through the separate merge launch (one workgroup per output row, the partials merged in
# split order): 18, 64, 512 and 1024 splits, verify rows on the MFMA kernel at 64, 32 and 18 splits, batch 3 with
# an idle user at 32 and 18 splits. Three calls give the same bits, match the oracle, leave the in-launch counters
# at zero and report nothing.
@pytest.mark.parametrize("B,ctx,T,pps", [(2, 1100, 1, 1), (1, 32768, 1, 8), (1, 32768, 1, 1), (1, 65536, 1, 1),
                                         (1, 8192, 4, 2), (3, 2000, 4, 1), (3, 1100, 4, 1)])  # fmt: skip
def test_many_splits_repeatable(dev, B, ctx, T, pps):
    d = W.attn_layer(B, ctx, "cpu", seed=3 * B + T + pps, T=T, num_blocks=B * (ctx // 64 + 1) + 64)
    if B == 3:
        d["seq_lens"][1] = 0  # idle: no workgroup of the user arrives at its counters
    g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
    mb = d["block_table"].shape[1]
    ws = torch.zeros(ops.lib().qs_paged_attention_workspace_bytes(B, T, 24, 4, 256, mb, pps), dtype=torch.uint8,
                     device=dev)  # fmt: skip
    st = ops.Status(dev)
    outs = []
    for _ in range(3):
        o = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"],
                                 pages_per_split=pps, ws=ws, status=st.word)  # fmt: skip
        torch.cuda.synchronize()
        assert int(ws[:CNT_BYTES].view(torch.int32).abs().sum()) == 0, "counters not re-armed"
        outs.append(o.cpu())
    assert st.peek() == 0
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[1], outs[2])
    ref = O.gqa_decode(d["q"], d["k_cache"], d["v_cache"], d["block_table"], d["seq_lens"], d["scale"])
    assert_attn_output(outs[0], O.bf16(ref))


@pytest.mark.parametrize("T", [1, 4])
def test_merge_launch_ragged(dev, T):
    """The merge launch over users of very different lengths: one user's 19 splits hold a single page of T rows
    among 18 empty splits (whose partials carry no weight), the other's all 19 pages."""
    d = W.attn_layer(2, 19 * 64, "cpu", seed=40 + T, T=T, num_blocks=64)
    d["seq_lens"] = torch.tensor([T, 19 * 64 - 5], dtype=torch.int32)
    o, o_ref, same = run_case(dev, d, pps=1)
    assert same
    assert_attn_output(o, o_ref)


@pytest.mark.parametrize("ctx,pps", [(131072, 64), (131072, 2), (262144, 4)])
def test_attention_long_context(dev, ctx, pps):
    """128k and 256k positions at batch 1 (the reference's published long-context decode points reach 256k):
    64 splits of 32 pages (of the 64 allowed), exactly the 1024-split limit, and 1024 splits at 256k."""
    d = W.attn_layer(1, ctx, "cpu", seed=ctx // 1024 + pps, num_blocks=ctx // 64 + 64)
    o, o_ref, same = run_case(dev, d, pps)
    assert same
    assert_attn_output(o, o_ref)


def test_attention_split_limits(dev):
    """More than 1024 splits or more than 64 pages per split are rejected before any launch."""
    d = W.attn_layer(1, 131072, dev, seed=1, num_blocks=2048 + 64)
    for pps in (1, 65):
        with pytest.raises(ValueError, match="splits|pages_per_split"):
            ops.paged_gqa_decode(d["q"], d["k_cache"], d["v_cache"], d["block_table"], d["seq_lens"], d["scale"],
                                 pages_per_split=pps)  # fmt: skip


def test_attention_negative_control(dev):
    """The check fails when the oracle drops the appended row (a missed append dependency)."""
    d = W.attn_layer(2, 40, "cpu", seed=12, num_blocks=64)  # 40 positions: the new row carries ~1/40 of the weight
    o, ref, _ = run_case(dev, d, 4)
    assert_attn_output(o, ref)
    wrong = O.bf16(O.gqa_decode(d["q"], d["k_cache"], d["v_cache"], d["block_table"], d["seq_lens"] - 1, d["scale"]))
    with pytest.raises(AssertionError):
        assert_attn_output(o, wrong)


# Query rows per KV head past one MFMA tile of the rows kernel's ranges: 33 .. 48 and 49 .. 64 in one block of 3 or 4
# tiles, 65 .. 96 and 97 .. 128 in two blocks; new rows that start a user's cache, end a page, cross pages and splits;
# one and two page groups; one split, in-range and past the last page.
@pytest.mark.parametrize(
    "G,T,lens,pps",
    [
        (6, 6, [6, 64, 700], 2),  # 36 rows; the first user holds nothing but its new rows
        (6, 8, [4099, 68, 1300], 8),  # 48 rows; new rows across pages, an odd page count per split
        (6, 8, [130], 1),  # one page per split
        (4, 13, [77, 640], 64),  # 52 rows, one split
        (8, 8, [8, 1027], 3),  # 64 rows
        (6, 11, [11, 138, 900], 2),  # 66 rows: two blocks of 3 tiles, 30 of them empty
        (6, 16, [1040, 16], 1),  # 96 rows; 16 new rows over two pages, each its own split
        (8, 13, [333], 4),  # 104 rows: two blocks of 4 tiles
        (8, 16, [72, 1999], 2),  # 128 rows, the most
    ],
)
@pytest.mark.parametrize("mixer", [False, True])
def test_verify_row_blocks(dev, G, T, lens, pps, mixer):
    B, nkv = len(lens), 4
    d = W.attn_layer(B, max(lens), "cpu", seed=G * 100 + T + pps, T=T, num_blocks=512)
    gen = torch.Generator().manual_seed(G + T)
    d["q"] = torch.randn(B, T, G * nkv, 256, generator=gen).bfloat16()
    d["seq_lens"] = torch.tensor(lens, dtype=torch.int32)
    if not mixer:
        o1, ref, same1 = run_case(dev, d, pps, fused=True)
        o2, _, same2 = run_case(dev, d, pps, fused=False)
        assert same1 and same2
        assert torch.equal(o1.cpu(), o2.cpu())
        assert_attn_output(o1, ref)
        return
    check_mixer(dev, d, pps, 64, gen)


def check_mixer(dev, d, pps, rot, gen, ws=None, close=assert_attn_output):
    """The mixer's call against the oracle: appended K rows within one bf16 ulp, V rows bit-exact, the output."""
    from conftest import bf16_ulp_mismatch

    T = d["q"].shape[1]
    gate = torch.randn(d["q"].shape, generator=gen).bfloat16()
    wq = (1 + 0.1 * torch.randn(256, generator=gen)) / 16.0
    wk = 1 + 0.1 * torch.randn(256, generator=gen)
    cos, sin = O.rope_tables((d["seq_lens"] - T)[:, None] + torch.arange(T)[None], rot) if rot else (None, None)
    g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
    tab = [t.to(dev) if rot else None for t in (cos, sin)]
    o = ops.attn_mixer_decode(g["q"], g["k_new"], g["v_new"], gate.to(dev), wq.to(dev), wk.to(dev), *tab, g["k_cache"],
                              g["v_cache"], g["block_table"], g["seq_lens"], pages_per_split=pps, rot=rot, ws=ws)  # fmt: skip
    kc, vc = d["k_cache"].clone(), d["v_cache"].clone()
    if not rot:
        cos, sin = torch.ones(*d["q"].shape[:2], 8), torch.zeros(*d["q"].shape[:2], 8)  # the identity rotation
    o_ref = O.attn_mixer(d["q"], d["k_new"], d["v_new"], gate, wq, wk, cos, sin, kc, vc, d["block_table"],
                         d["seq_lens"], rot=rot or 16)  # fmt: skip
    assert torch.equal(g["v_cache"].cpu(), vc)
    ulps, frac = bf16_ulp_mismatch(g["k_cache"].cpu(), kc)
    assert ulps <= 1 and frac < 1e-3, (ulps, frac)
    close(o, o_ref)


# The mixer's new rows, normalised, rotated and staged before the page loop: one and two tokens (held in LDS), three
# and more (the rows kernel), a page per split or two in one (test_page_groups walks more); a user with only its new rows, rows
# that end, start and cross a page; every rotation width.
@pytest.mark.parametrize("T,lens,pps", [(1, [1, 64, 65, 700], 8), (1, [65, 128], 1), (2, [2, 65, 333], 4),
                                        (2, [129, 64], 1), (4, [66, 4], 2), (4, [193], 1)])  # fmt: skip
@pytest.mark.parametrize("rot", [0, 16, 256])
def test_mixer_new_rows(dev, T, lens, pps, rot):
    d = W.attn_layer(len(lens), max(lens), "cpu", seed=T + pps + rot, T=T, num_blocks=64)
    d["seq_lens"] = torch.tensor(lens, dtype=torch.int32)
    check_mixer(dev, d, pps, rot, torch.Generator().manual_seed(T + rot))


def test_verify_row_blocks_idle_and_bad_page(dev):
    """Two row blocks with an idle user and a page entry outside the pool: the idle user's rows are zero, the bad
    page is reported and not attended, the others match the oracle."""
    T, lens = 11, [500, 3, 900]
    d = W.attn_layer(3, 900, "cpu", seed=7, T=T, num_blocks=64)
    d["seq_lens"] = torch.tensor(lens, dtype=torch.int32)
    o_ref = O.bf16(O.gqa_decode(d["q"], d["k_cache"], d["v_cache"], d["block_table"], d["seq_lens"], d["scale"]))
    g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
    g["block_table"][2, 5] = 64
    st = ops.Status(dev)
    o = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"],
                             pages_per_split=2, status=st.word)  # fmt: skip
    assert st.peek() == ops.STATUS_PAGE
    assert_attn_output(o[0], o_ref[0])
    assert int(o[1].count_nonzero()) == 0
    keep = torch.ones(900, dtype=torch.bool)
    keep[5 * 64 : 6 * 64] = False
    rows = d["block_table"][2, :15].long()
    K, V = (d[n][rows].permute(1, 0, 2, 3).reshape(4, -1, 256)[:, :900].float() for n in ("k_cache", "v_cache"))
    for t in range(T):
        seen = keep & (torch.arange(900) <= 900 - T + t)
        s = (d["q"][2, t].float().view(4, 6, 256) @ K[:, seen].transpose(1, 2)) * d["scale"]
        assert_attn_output(o[2, t].view(4, 6, 256), O.bf16(s.softmax(-1) @ V[:, seen]))


# A step of 3 or more tokens with at most 16 query rows per KV head stores its new rows first and reads the pages they
# lie in again. A grid of at most 256 workgroups walks one page each though the caller allows two (2 users x 4 KV heads
# x 4 pages), where K is read in the score operand's layout; 66 users x 4 KV heads are past that and walk the caller's
# two pages at a time. The new rows cross a page, end one, fill a user's cache or start it.
@pytest.mark.parametrize("G,T", [(4, 3), (4, 4), (2, 3), (2, 8), (1, 3), (1, 16)])
@pytest.mark.parametrize("B,pps", [(2, 1), (2, 2), (66, 2)])
@pytest.mark.parametrize("mixer", [False, True])
def test_few_rows_append(dev, G, T, B, pps, mixer):
    gen = torch.Generator().manual_seed(G * 100 + T + B)
    d = W.attn_layer(B, 256, "cpu", seed=G * 100 + T + pps, T=T, num_blocks=B * 4 + 8)
    d["q"] = torch.randn(B, T, G * 4, 256, generator=gen).bfloat16()
    d["seq_lens"] = torch.tensor(([130, 256] + [T, 64, 65, 192] * 16)[:B], dtype=torch.int32)
    assert plan(B, T, G, 4, pps, mixer)[0] == (2 if B == 66 else 1)
    if mixer:
        return check_mixer(dev, d, pps, 64, gen)
    o1, ref, same1 = run_case(dev, d, pps, fused=True)
    o2, _, same2 = run_case(dev, d, pps, fused=False)
    assert same1 and same2
    assert torch.equal(o1.cpu(), o2.cpu())
    assert_attn_output(o1, ref)


# The rows kernel's forms for up to 8 new tokens and for up to 16, 2, 3 and 4 query tiles each side of 8: 32 and 18 rows,
# 48 and 36, 64 and 54 (the longest call of 8 tokens, the shortest past it). A table of 5 pages is walked a page per
# workgroup, one of 2 pages whole (both at once where there is room); new rows fill a user's cache, cross a page, end one.
@pytest.mark.parametrize("G,T", [(4, 8), (2, 9), (6, 8), (4, 9), (8, 8), (6, 9)])
@pytest.mark.parametrize("width", [5, 2])
@pytest.mark.parametrize("mixer", [False, True])
def test_verify_token_forms(dev, G, T, width, mixer):
    lens = [T, 64 + T // 2, width * 64]
    assert plan(3, T, G, width, 8, mixer)[0] == (2 if width == 2 and pairs(T, G, mixer) else 1)
    d = W.attn_layer(3, width * 64, "cpu", seed=G + T, T=T, num_blocks=32)
    gen = torch.Generator().manual_seed(G + T)
    d["q"] = torch.randn(3, T, G * 4, 256, generator=gen).bfloat16()
    d["seq_lens"] = torch.tensor(lens, dtype=torch.int32)
    if mixer:
        return check_mixer(dev, d, 8, 64, gen)
    o, ref, same = run_case(dev, d, 8)
    assert same
    assert_attn_output(o, ref)


# A table wider than its users: the splits past a user's pages write no partial, and the merges read none of theirs (the
# workspace holds NaNs); table entries past a user's pages are not looked at. Merged in the launch (4 and 8 splits) and in
# one of their own (16 to 24, and 65, past one load of every split's maximum); users of one page, of all, idle.
@pytest.mark.parametrize("B,T,width,pps,merged", [(16, 1, 16, 4, True), (8, 2, 16, 2, True), (3, 1, 144, 8, False),
                                                  (5, 2, 24, 1, False), (4, 4, 64, 8, False), (3, 8, 130, 2, False),
                                                  (3, 11, 40, 2, False)])  # fmt: skip
@pytest.mark.parametrize("mixer", [False, True])
def test_wide_tables(dev, B, T, width, pps, merged, mixer):
    assert plan(B, T, 6, width, pps, mixer)[2] == merged
    d = W.attn_layer(B, width * 64, "cpu", seed=B + T + width, T=T, num_blocks=B * width + 8)
    idle = 0 if not mixer else T  # the oracle's mixer has no idle users
    d["seq_lens"] = torch.tensor(([T, width * 64, idle, 65, 64] + [128 + T] * B)[:B], dtype=torch.int32)
    for b in range(B):
        d["block_table"][b, -(-int(d["seq_lens"][b]) // 64) :] = -1
    ws = torch.zeros(ops.lib().qs_paged_attention_workspace_bytes(B, T, 24, 4, 256, width, pps), dtype=torch.uint8,
                     device=dev)  # fmt: skip
    ws[CNT_BYTES:] = 0xFF
    if mixer:
        check_mixer(dev, d, pps, 64, torch.Generator().manual_seed(width), ws=ws)
    else:
        g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
        st = ops.Status(dev)
        o = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"],
                                 pages_per_split=pps, ws=ws, status=st.word)  # fmt: skip
        assert st.peek() == 0
        live = [b for b in range(B) if b != 2]
        ref = O.gqa_decode(d["q"][live], d["k_cache"], d["v_cache"], d["block_table"][live], d["seq_lens"][live], d["scale"])
        assert_attn_output(o[live], O.bf16(ref))
        assert int(o[2].count_nonzero()) == 0
    assert int(ws[:CNT_BYTES].view(torch.int32).abs().sum()) == 0, "counters not re-armed"


# A call that fits one split needs no workspace: the library writes nothing to one that is given (here full of 0xFF, where
# counters would have to be zero), and the ops take one too small for finer splits as they take none.
@pytest.mark.parametrize("T", [1, 4])
def test_one_split_leaves_the_workspace(dev, T):
    import ctypes

    d = W.attn_layer(2, 4 * 64, "cpu", seed=T, T=T, num_blocks=16)
    g = {k: (v.to(dev) if torch.is_tensor(v) else v) for k, v in d.items()}
    L = ops.lib()
    nbytes = L.qs_paged_attention_workspace_bytes(2, T, 24, 4, 256, 4, 8)
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=dev)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    o = torch.empty_like(g["q"])
    assert L.qs_paged_gqa_decode(p(g["q"]), None, None, p(g["k_cache"]), p(g["v_cache"]), p(g["block_table"]),
                                 p(g["seq_lens"]), p(o), p(ws), 2, T, 24, 4, 256, 64, 4, 16, 8, d["scale"], None,
                                 torch.cuda.current_stream().cuda_stream) == 0  # fmt: skip
    ref = O.bf16(O.gqa_decode(d["q"], d["k_cache"], d["v_cache"], d["block_table"], d["seq_lens"], d["scale"]))
    assert_attn_output(o, ref)
    assert int((ws != 0xFF).sum()) == 0
    o2 = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"], ws=ws[:256])
    none = ops.paged_gqa_decode(g["q"], g["k_cache"], g["v_cache"], g["block_table"], g["seq_lens"], d["scale"])
    assert torch.equal(o2, o) and torch.equal(none, o)
    check_mixer(dev, d, 8, 64, torch.Generator().manual_seed(T), ws=ws[:256])
    assert int((ws != 0xFF).sum()) == 0


def assert_users(o, ref):
    """Each user's output against its own RMS: a probability rounded to bf16 is off by 2^-9 / sqrt(3) of itself (RMS), so an
    output by 1.1e-3 of the user's RMS, a ninth of the floor; a short user's RMS is many times that of a long batch."""
    for a, b in zip(o, ref):
        assert_attn_output(a, b)


# 70 users x 4 KV heads, past a workgroup per CU, walk the caller's pages. One page group against two in the rows kernel, by
# its tiles, the pages and the mixer, for up to 8 new tokens and more: 2 tiles at 4 and 5 pages, 3 and 4 tiles at 2 and 3,
# with the mixer 2 tiles at 2 (in 2 splits, whole) and 3, 3 at 2; and the mixer's one- and two-token calls, two at a time.
@pytest.mark.parametrize("G,T,width,pps,mixer", [
    (6, 4, 8, 4, False), (6, 4, 10, 5, False), (2, 9, 10, 5, False), (6, 8, 4, 2, False), (6, 8, 6, 3, False),
    (4, 9, 6, 3, False), (8, 8, 6, 3, False), (4, 13, 6, 3, False), (6, 4, 4, 2, True), (6, 4, 2, 2, True), (6, 4, 6, 3, True),
    (2, 9, 6, 3, True), (6, 8, 4, 2, True), (6, 1, 7, 5, True), (6, 2, 7, 5, True),
])  # fmt: skip
def test_page_groups(dev, G, T, width, pps, mixer):
    B = 70
    assert plan(B, T, G, width, pps, mixer)[0] == pps
    d = W.attn_layer(B, width * 64, "cpu", seed=G + T + width, T=T, num_blocks=B * width + 8)
    gen = torch.Generator().manual_seed(G + T)
    d["q"] = torch.randn(B, T, G * 4, 256, generator=gen).bfloat16()
    d["seq_lens"] = torch.randint(T, width * 64 + 1, (B,), generator=gen).to(torch.int32)
    if mixer:
        return check_mixer(dev, d, pps, 64, gen, close=assert_users)
    o, ref, same = run_case(dev, d, pps)
    assert same
    assert_users(o, ref)
