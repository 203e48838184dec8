"""Prefill blocks that split the keys over groups of waves (grids that leave CUs idle).

Lengths around the 64-key tile and the groups' turns (a last group with no tile, a single
partial tile, diagonal tiles on another group than the walk's first), both masks, padded head
dims, both row orders, int8 rows, and V scales that need the fp16 range shift (2^E > 1).
Against the float64 oracle with the attention bars of helpers.py.
"""
import numpy as np
import pytest
import torch

import workloads
from helpers import assert_attn_close
from oracle import oracle_c

pytestmark = pytest.mark.gpu


def _np(t):
    return t.detach().cpu().numpy()


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
