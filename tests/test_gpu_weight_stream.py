"""Weight-streaming projections and the MLP half on the GPU against the oracle: the device quantizer bit for
bit against the oracle's MXFP4 / MXFP8 / MXINT8 quantization and layout (ties, saturation, zero and tiny
blocks), the streamed y = h W against h times the dequantized weight (fp32 accumulation: rtol 1e-4), the MLP
half x + bf16(silu(h G) (h U)) D at the reference's shape (H 5120, I 17408) and at small ones, and the MLP half
with MXINT8 down weights against unquantized fp32 down weights (the reference's 8-bit precision)."""
import math

import numpy as np
import pytest
import torch

from oracle import weight_stream as WS
from qwen36_state import ops

pytestmark = pytest.mark.gpu


def _rand(shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g) * scale


def _special_blocks(w, fmt):
    """Blocks that exercise the encoder's edges: all zeros, exact ties at scale 1, saturation, tiny values."""
    w[:32, 0] = 0.0
    if fmt == 4:
        ties = [6.0, 0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0, -0.3, 0.1, -0.1, -6.0, 0.5, -2.5, -5.0]
        w[32:64, 1] = 0.0
        w[32 : 32 + len(ties), 1] = torch.tensor(ties)
        w[64:96, 2] = torch.linspace(-7.9, 7.9, 32)
    elif fmt == 8:
        ties = [480.0, 448.0, 1.0, 1.0625, 1.1875, 2.0**-10, 3 * 2.0**-10, -1.0, 2.0**-6, -1.0625, 300.0]
        w[32:64, 1] = 0.0
        w[32 : 32 + len(ties), 1] = torch.tensor(ties)
        w[64:96, 2] = torch.linspace(-500.0, 500.0, 32)
    else:  # MXINT8 at scale 1: codes round(64 v), ties to even, saturating at +-127
        ties = [1.984375, 1.0, 0.5, -1.0, 1.999, -1.999, 2.0**-7, 3 * 2.0**-7, -3 * 2.0**-7, 0.3, -5 * 2.0**-7]
        w[32:64, 1] = 0.0
        w[32 : 32 + len(ties), 1] = torch.tensor(ties)
        w[64:96, 2] = torch.linspace(-3.9, 3.9, 32)
    w[96:128, 3] = 1e-30 * torch.arange(1, 33)
    return w


@pytest.mark.parametrize("fmt", [4, 8, 9])
def test_quantize_matches_oracle(dev, fmt):
    K, N = 256, 64
    w = _special_blocks(_rand((K, N), 1, 0.05), fmt)
    packed = ops.MxWeight.quantize(w.to(dev), fmt).packed.cpu().numpy()
    codes, e = WS.mx_quantize(w.double(), fmt)
    np.testing.assert_array_equal(packed, WS.mx_pack(codes, e, fmt))


def _dequantized(W):
    codes, e = WS.mx_unpack(W.packed.cpu().numpy(), W.K, W.N, W.fmt)
    return WS.mx_dequantize(codes, e, W.fmt)


# K splits (one row up to 7 (MXFP4) / 15 (MXFP8) rows: the rows a workgroup stages must fit in 24 KB of LDS;
# more rows: read from L2 with each weight group; then more splits while the grid is small): 1 for
# (4, 512, 128, 1); 16 for (8, 17408, 64, 1), summed over 2 round trips of the last workgroup; 16 for
# (8, 17408, 64, 16) and 2 for (4, 5120, 256, 8) and (4, 5120, 32, 13) with rows from L2
@pytest.mark.parametrize("fmt,K,N,B", [(4, 512, 128, 1), (4, 5120, 256, 8), (8, 1024, 64, 16), (8, 17408, 64, 1),
                                       (4, 256, 2048, 3), (8, 17408, 64, 16), (4, 5120, 32, 13), (9, 17408, 64, 1),
                                       (9, 1024, 64, 16), (9, 5120, 256, 3)])  # fmt: skip
def test_mx_linear(dev, fmt, K, N, B):
    w = _rand((K, N), 2, 1 / math.sqrt(K))
    W = ops.MxWeight.quantize(w.to(dev), fmt)
    h = _rand((B, K), 3).bfloat16()
    y = ops.mx_linear(h.to(dev), W)
    ref = h.double() @ _dequantized(W)
    torch.testing.assert_close(y.cpu().double(), ref, rtol=1e-4, atol=1e-5 * ref.abs().max().item())
    # the split sums are re-armed by each launch: a second call gives the same bits
    assert torch.equal(ops.mx_linear(h.to(dev), W), y)


def _mlp(dev, B, H, I, seed=4, down_fmt=ops.MXINT8):
    gate = ops.MxWeight.quantize(_rand((H, I), seed, 1 / math.sqrt(H)).to(dev), ops.MXFP4)
    up = ops.MxWeight.quantize(_rand((H, I), seed + 1, 1 / math.sqrt(H)).to(dev), ops.MXFP4)
    down = ops.MxWeight.quantize(_rand((I, H), seed + 2, 0.5 / math.sqrt(I)).to(dev), down_fmt)
    gamma = 1 + 0.1 * _rand((H,), seed + 3)
    x = _rand((B, H), seed + 4)
    return x, gamma, gate, up, down


def _rel(a, b):
    return ((a - b).norm() / b.norm()).item()


# the last workgroup of a block applying silu after K splits: (16, 5120, 1024) gate | up in 4 splits,
# (4, 5120, 2048) in 2; (1, 10240, 512): one row too long for the gate | up workgroups to normalise, through the
# rmsnorm kernel's two passes over 8192-value chunks
# column blocks and K splits: (2, 128, 64) one group for 8 waves; (16, 5120, 10240) 4 tiles per block, gate | up whole,
# down in 3 splits; (2, 2560, 17088) 2 tiles per block, 512 blocks whole and 22 in 2 splits, down 4 tiles in 6 splits;
# (3, 4096, 16448) 4 tiles per block, 256 blocks whole and one in 4 splits; (2, 2176, 4224) 1 tile per block, 256 whole
# and 8 in 2 splits; (1, 6144, 1024) the longest row gate | up workgroups normalise, (1, 6272, 512) the first past it
@pytest.mark.parametrize("B,H,I,fmt", [(2, 128, 64, 9), (1, 128, 64, 9), (16, 5120, 10240, 9), (2, 2560, 17088, 8),
                                       (1, 6144, 1024, 9), (1, 6272, 512, 9), (1, 256, 512, 9), (8, 512, 1024, 9), (16, 256, 256, 9), (1, 5120, 17408, 9),
                                       (16, 5120, 1024, 9), (5, 1024, 2048, 9), (4, 5120, 2048, 9), (1, 10240, 512, 9),
                                       (1, 5120, 17408, 8), (16, 256, 256, 8), (4, 5120, 2048, 8),
                                       (3, 4096, 16448, 9), (2, 2176, 4224, 8)])  # fmt: skip
def test_mlp_decode(dev, B, H, I, fmt):
    x, gamma, gate, up, down = _mlp(dev, B, H, I, down_fmt=fmt)
    out = ops.mlp_decode(x.to(dev), gamma.to(dev), gate, up, down).cpu().double()
    G, U, D = _dequantized(gate), _dequantized(up), _dequantized(down)
    ref = WS.mlp_half(x.double(), gamma.double(), G, U, D)
    delta, dref = out - x.double(), ref - x.double()
    # h and z are bf16: where the kernel's fp32 rmsnorm or gate product sits within an ulp of a bf16 rounding
    # boundary it may round the other way; such elements move the output by ~2^-9 of one term
    assert _rel(delta, dref) < 2e-3
    torch.testing.assert_close(delta, dref, rtol=2e-2, atol=5e-3 * dref.pow(2).mean().sqrt().item())
    # negative control: the oracle with gate and up exchanged is far off
    assert _rel(delta, WS.mlp_half(x.double(), gamma.double(), U, G, D) - x.double()) > 0.1


# B = 1 takes the path where the gate | up workgroups normalise x themselves while down workgroups of the
# same launch store x_out: in place, no x_out store may land before every x read
@pytest.mark.parametrize("B,H,I", [(4, 256, 512), (1, 5120, 17408)])
def test_mlp_decode_in_place_and_repeatable(dev, B, H, I):
    x, gamma, gate, up, down = _mlp(dev, B, H, I, seed=9)
    xd = x.to(dev)
    a = ops.mlp_decode(xd, gamma.to(dev), gate, up, down)
    b = xd.clone()
    ops.mlp_decode(b, gamma.to(dev), gate, up, down, out=b)
    assert torch.equal(a, b)


# gamma None: the norm weight folded into the rows of gate and up, as the reference's weights.py:107-112 loads
# them; one row (rmsnorm inside the gate | up launch) and eight (its own launch)
@pytest.mark.parametrize("B", [1, 8])
def test_mlp_decode_folded_gamma(dev, B):
    x, gamma, gate, up, down = _mlp(dev, B, 512, 1024, seed=12)
    out = ops.mlp_decode(x.to(dev), None, gate, up, down).cpu().double()
    G, U, D = _dequantized(gate), _dequantized(up), _dequantized(down)
    ref = WS.mlp_half(x.double(), None, G, U, D)
    assert _rel(out - x.double(), ref - x.double()) < 2e-3
    assert torch.equal(ops.mlp_decode(x.to(dev), torch.ones(512, device=dev), gate, up, down).cpu().double(), out)


@pytest.mark.parametrize("B", [1, 4])
def test_mlp_down_precision_against_fp32_weights(dev, B):
    """The MLP half with the down weight in MXINT8 against the same half with the unquantized fp32 down weight
    (gate | up dequantized from MXFP4 on both sides): the quantization of down moves the MLP's delta by 0.8%
    (RMS-relative, H 512, I 2048; the oracle alone gives 0.78%), the bound here 1.2%. The same weight in
    MXFP8 (E4M3, 3 mantissa bits) moves it by ~3%: MXINT8 is the format with the reference's 7-bit precision."""
    H, I = 512, 2048
    d32 = _rand((I, H), 6, 0.5 / math.sqrt(I))
    res = {}
    for fmt in (ops.MXINT8, ops.MXFP8):
        x, gamma, gate, up, _ = _mlp(dev, B, H, I)
        down = ops.MxWeight.quantize(d32.to(dev), fmt)
        out = ops.mlp_decode(x.to(dev), gamma.to(dev), gate, up, down).cpu().double()
        ref = WS.mlp_half(x.double(), gamma.double(), _dequantized(gate), _dequantized(up), d32.double())
        res[fmt] = _rel(out - x.double(), ref - x.double())
    assert res[ops.MXINT8] < 1.2e-2, res
    assert res[ops.MXFP8] > 2e-2, res


def test_rejects_bad_shapes(dev):
    with pytest.raises(ValueError):
        ops.MxWeight.quantize(torch.zeros(100, 16, device=dev), ops.MXFP4)
    with pytest.raises(ValueError):
        ops.MxWeight.quantize(torch.zeros(128, 20, device=dev), ops.MXFP8)
    W = ops.MxWeight.quantize(torch.zeros(128, 16, device=dev), ops.MXFP4)
    with pytest.raises(ValueError):
        ops.mx_linear(torch.zeros(17, 128, dtype=torch.bfloat16, device=dev), W)
    x, gamma, gate, up, down = _mlp(dev, 2, 256, 512)
    with pytest.raises(ValueError):
        ops.mlp_decode(x.to(dev), gamma.to(dev), up, gate, gate)  # down must be MXINT8 or MXFP8 [I, H]
