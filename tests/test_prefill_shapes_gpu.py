"""Prefill blocks that split the keys over groups of waves (grids that leave CUs idle).

Lengths around the 64-key tile and the groups' turns (a last group with no tile, a single
partial tile, diagonal tiles on another group than the walk's first), both masks, padded head
dims, both row orders, int8 rows, and V scales that need the fp16 range shift (2^E > 1).
Against the float64 oracle with the attention bars of helpers.py, and against the same heads
on the shape with one group.
"""
import numpy as np
import pytest
import torch

import int8k_capi as capi
import workloads
from helpers import assert_attn_close
from oracle import oracle_c

pytestmark = pytest.mark.gpu


def _np(t):
    return t.detach().cpu().numpy()


# (D, BH, S, causal) -> (query waves, key groups): every instance of the kernel with and
# without the mask, on whole and padded head dims
GROUPED = [
    (64, 12, 449, False, (2, 4)), (48, 12, 449, False, (2, 4)), (64, 12, 384, True, (2, 4)),
    (32, 12, 385, True, (2, 4)), (64, 24, 1030, False, (4, 2)), (48, 24, 1030, False, (4, 2)),
    (64, 24, 1030, True, (4, 2)), (48, 24, 1023, True, (4, 2)), (128, 12, 449, False, (2, 2)),
    (80, 12, 449, False, (2, 2)), (128, 12, 127, True, (2, 2)), (96, 12, 126, True, (2, 2)),
    (128, 32, 641, False, (4, 2)), (80, 32, 641, False, (4, 2)), (128, 12, 1030, True, (4, 2)),
    (80, 12, 1023, True, (4, 2))]
ONE_GROUP = [
    (64, 128, 641, False, (4, 1)), (48, 128, 641, True, (4, 1)), (64, 128, 449, True, (4, 1)),
    (48, 128, 450, False, (4, 1)), (128, 128, 641, False, (8, 1)), (128, 128, 450, True, (8, 1)),
    (112, 128, 449, True, (8, 1)), (80, 128, 449, False, (8, 1))]


def _rows(shape, g, outliers):
    """Quantized N(0, 1) rows, with `outliers` 1% of the channels x8: scores spread over tens
    of powers of two, so that tiles past the first raise the running maximum."""
    x = torch.randn(shape, generator=g)
    if outliers:
        x[..., torch.randperm(shape[-1], generator=g)[:max(1, shape[-1] // 100)]] *= 8.0
    s = x.abs().amax(-1).clamp(min=1e-8) / 127.0
    return (x / s.unsqueeze(-1)).round().clamp(-128, 127).to(torch.int8), s


def _case(BH, S, D, seed, outliers, device):
    g = torch.Generator().manual_seed(seed)
    return [t.to(device) for n in range(3) for t in _rows((1, BH, S, D), g, outliers and n < 2)]


def _forward(ext, c, causal):
    q, sq, k, sk, v, sv = c
    return ext.int8_attention_forward(q, k, v, sq, sk, sv, is_causal=causal)


@pytest.mark.parametrize("D,BH,S,causal,shape", GROUPED + ONE_GROUP)
def test_every_shape_matches_the_oracle(ext, gpu, D, BH, S, causal, shape):
    assert capi.attention_block_shape(BH, S, D, causal) == shape
    c = _case(BH, S, D, seed=S + D, outliers=False, device=gpu)
    out = _forward(ext, c, causal)
    torch.cuda.synchronize()
    heads = [0, BH // 2, BH - 1]
    q, sq, k, sk, v, sv = (_np(t[0, heads]) for t in c)
    ref = oracle_c.prefill_attention(q, k, v, sq, sk, sv, causal=causal)
    assert_attn_close(_np(out[0, heads].float()), ref, f"D{D} BH{BH} S{S} causal {causal}")


@pytest.mark.parametrize("negative", [False, True])
@pytest.mark.parametrize("D,BH,S,causal,shape", GROUPED)
def test_groups_match_one_group(ext, gpu, D, BH, S, causal, shape, negative):
    # The same heads in a batch that fills the GPU run with one group.  The fp16 probabilities
    # are rounded against the same running maximum, so the two differ by the order of fp32 sums
    # (about S / 16 additions of 2^-24 each, of terms up to max |v|, on both sides) and at most
    # one step of the fp16 output, on the few rows where that moves it across a rounding.
    assert capi.attention_block_shape(BH, S, D, causal) == shape
    # (no batch of causal prompts up to 128 long runs with one group: they are taken as the
    # first rows of longer prompts there, which no later key reaches)
    S1 = S + 322 if causal and S <= 128 else S
    times = next(r for r in range(2, 129)
                 if capi.attention_block_shape(BH * r, S1, D, causal)[1] == 1)
    c = _case(BH, S1, D, seed=S + D, outliers=True, device=gpu)
    if negative:  # negative query scales: every tile sets the maximum
        c[1][..., ::3] *= -1
    small = _forward(ext, [t[:, :, :S].contiguous() for t in c], causal)
    large = _forward(ext, [torch.cat([t] * times) for t in c], causal)
    torch.cuda.synchronize()
    a, b = _np(small[0].double()), _np(large[times - 1, :, :S].double())
    vmax = float((c[4].float().abs().amax(-1) * c[5]).max())
    bound = 2.0 ** -10 * np.abs(b) + 2 * (S / 16 + 8) * 2.0 ** -24 * vmax
    assert np.all(np.abs(a - b) <= bound), (np.abs(a - b) - bound).max()
    assert (a != b).mean() <= 0.02, (a != b).mean()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [48, 64, 80, 128])
@pytest.mark.parametrize("S", [65, 127, 193, 257, 448, 641, 1030])
def test_split_keys(ext, gpu, S, D, causal):
    B, H = 2, 2
    p = workloads.prefill_case(B, H, S, D, seed=S + D, device=gpu, gen_device="cpu")
    if S == 257:
        # 127 max(sV) = 50800: above the 32768 that needs no shift (E = 1), and below 65504,
        # so that no output row, a weighted mean of V rows, leaves the fp16 range
        p["sV"] = p["sV"] * 400.0 / p["sV"].max()
    args = [p[k] for k in ("Qi", "Ki", "Vi", "sQ", "sK", "sV")]
    out = ext.int8_attention_forward(*args, is_causal=causal, out_bshd=True)
    q, s = ext.int8_attention_forward_quant(*args, is_causal=causal)
    plain = ext.int8_attention_forward(*args, is_causal=causal)
    rq, rs = ext.quantize_per_token(plain)
    torch.cuda.synchronize()
    assert torch.equal(out, plain.transpose(1, 2)) and torch.equal(q, rq) and torch.equal(s, rs)
    ref = oracle_c.prefill_attention(*(_np(t).reshape(B * H, S, D) for t in args[:3]),
                                     *(_np(t).reshape(B * H, S) for t in args[3:]), causal=causal)
    got = _np(plain.float()).reshape(B * H, S, D)
    if S == 257:  # outputs of thousands: the bars of a V scale of one
        scale = float(np.abs(ref).max())
        got, ref = got / scale, ref / scale
    assert_attn_close(got, ref, f"S{S} D{D} causal {causal}")


def test_split_keys_masked_rows_are_finite(ext, gpu):
    # scores far apart between the groups: a group whose keys all lose merges with weight 0
    B, H, S, D = 1, 2, 512, 64
    p = workloads.prefill_case(B, H, S, D, seed=7, device=gpu, gen_device="cpu")
    p["sK"][..., 64:128] *= 300.0
    args = [p[k] for k in ("Qi", "Ki", "Vi", "sQ", "sK", "sV")]
    for causal in (False, True):
        out = ext.int8_attention_forward(*args, is_causal=causal)
        torch.cuda.synchronize()
        ref = oracle_c.prefill_attention(*(_np(t).reshape(B * H, S, D) for t in args[:3]),
                                         *(_np(t).reshape(B * H, S) for t in args[3:]),
                                         causal=causal)
        assert_attn_close(_np(out.float()).reshape(B * H, S, D), ref, f"causal {causal}")
