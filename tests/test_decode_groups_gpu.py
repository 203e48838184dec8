"""Decode plans of several blocks per (b,h): partials merged by the combine kernel.

Shapes sit at the edges of the layout: one row past a whole wave iteration, odd row
strides at D = 64 (the paired rows count from the row before a head that starts in the
middle of a 128-byte line), a cache longer than the sequence, chunks that end inside an
iteration, empty tail blocks, and the same calls without a workspace.  Against float64 attention with fp32 sums' bound: the fp16 rounding of the
output (2^-11 relative) plus the 2e-3 that the fp32 softmax over up to 2^15 rows moves.
"""
import ctypes

import numpy as np
import pytest
import torch

import int8k_capi as capi
import workloads
from helpers import assert_attn_close

pytestmark = pytest.mark.gpu


def _ref(c, S):
    q = c["Qi"].double() * c["sQ"].double().unsqueeze(-1)
    k = c["Ki"][:, :, :S].double() * c["sK"][:, :, :S].double().unsqueeze(-1)
    v = c["Vi"][:, :, :S].double() * c["sV"][:, :, :S].double().unsqueeze(-1)
    s = (k * q.unsqueeze(2)).sum(-1) * q.shape[-1] ** -0.5
    return (torch.softmax(s, -1).unsqueeze(-1) * v).sum(2).cpu().numpy()


def _decode(c, S, ws):
    """Status and rows of the cache entry with the workspace tensor `ws` (None: a null one)."""
    B, H, cap, D = c["Ki"].shape
    out = torch.empty((B * H, D), dtype=torch.float16, device=c["Ki"].device)
    st = capi.load().int8k_decode_attention_forward_cache(
        *(ctypes.c_void_p(t.data_ptr()) for t in (c["Qi"], c["Ki"], c["Vi"], out, c["sQ"],
                                                  c["sK"], c["sV"])),
        B * H, S, cap, D, 0, ctypes.c_void_p(0 if ws is None else ws.data_ptr()),
        0 if ws is None else ws.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return st, out.float().reshape(B, H, D).cpu().numpy()


# null: what a call without a workspace does: "none" is needed, it falls back to "one" block per
# (b,h), or it is refused (a plan of more than 16 chunks that never merged on chip)
@pytest.mark.parametrize("B,H,D,S,cap,null", [
    (1, 3, 64, 4097, 4097, "refused"), (1, 5, 64, 8191, 8191, "refused"),
    (2, 3, 64, 5000, 5001, "refused"), (1, 12, 64, 6000, 6000, "refused"),
    (2, 2, 128, 12001, 12288, "refused"), (1, 12, 64, 4096, 4096, "one"),
    (1, 3, 128, 2113, 2113, "one"), (1, 1, 128, 1600, 1601, "one"), (4, 16, 128, 2000, 2001, "one"),
    (1, 2, 64, 33, 37, "none"), (1, 3, 64, 2049, 2050, "none"), (3, 7, 64, 63, 63, "none"),
    (1, 300, 64, 515, 515, "none"), (5, 60, 128, 3001, 3001, "none")])
def test_grouped_plans_match_float64(gpu, B, H, D, S, cap, null):
    c = workloads.decode_case(B, H, D, cap, seed=S, device=gpu, outlier_frac=0.01)
    n = capi.decode_workspace_bytes(B * H, S, D)
    assert (n == 0) == (null == "none")
    ref = _ref(c, S)
    label = f"{B} {H} {D} {S} {cap}"
    st, out = _decode(c, S, torch.empty(max(n, 1), dtype=torch.uint8, device=gpu))
    assert st == capi.INT8K_OK
    assert_attn_close(out, ref, label)
    # no workspace, and one byte less than the plan's partials
    for ws in [None] + ([torch.empty(n - 1, dtype=torch.uint8, device=gpu)] if n else []):
        st, out = _decode(c, S, ws)
        if null == "refused":
            assert st == capi.INT8K_ERR_WORKSPACE
        else:
            assert st == capi.INT8K_OK
            assert_attn_close(out, ref, label)


@pytest.mark.parametrize("D,S", [(64, 130), (128, 130), (64, 400), (128, 64), (64, 1)])
def test_infinite_value_scale_stays_in_its_dims(gpu, D, S):
    # fewer chunks than the block kernel's 8 waves: the absent ones add nothing, also where
    # a present one holds infinities (inf, with the sign of v, and NaN only where v is 0)
    c = workloads.decode_case(1, 3, D, S, seed=D + S, device=gpu, outlier_frac=0.0)
    assert capi.decode_num_splits(3, S, D) < 8
    c["sV"][..., S - 1] = float("inf")
    st, out = _decode(c, S, None)
    assert st == capi.INT8K_OK
    v = c["Vi"][:, :, S - 1].cpu().numpy().astype(np.float64)
    with np.errstate(invalid="ignore"):
        np.testing.assert_array_equal(out, v * np.inf)


@pytest.mark.parametrize("D,page,lens", [(64, 16, [6000, 1, 17, 3000]), (128, 64, [9000, 65]),
                                         (64, 1024, [5001, 0]), (128, 16, [20000])])
def test_grouped_paged_plans_match_float64(gpu, D, page, lens):
    H = 4
    c = workloads.paged_case(len(lens), H, D, page, lens, seed=page + D, device=gpu)
    out = capi.decode_attention_paged(c["Qi"], c["K_pages"], c["V_pages"], c["sQ"],
                                      c["sK_pages"], c["sV_pages"], c["block_tables"],
                                      c["context_lens"], c["max_context"])
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        o = out[b].float().cpu().numpy()
        if n == 0:
            assert np.all(o == 0)
            continue
        t = c["block_tables"][b, :-(-n // page)].long()
        flat = {k: c[k][t].transpose(0, 1).reshape(H, len(t) * page, -1)[:, :n]
                for k in ("K_pages", "V_pages", "sK_pages", "sV_pages")}
        ref = _ref(dict(Qi=c["Qi"][b:b + 1], sQ=c["sQ"].reshape(len(lens), H)[b:b + 1],
                        Ki=flat["K_pages"][None], Vi=flat["V_pages"][None],
                        sK=flat["sK_pages"][None, ..., 0], sV=flat["sV_pages"][None, ..., 0]), n)
        assert_attn_close(o, ref[0], f"paged D{D} page{page} len{n}")


@pytest.mark.parametrize("D,H,page,longest", [(64, 32, 64, 600), (64, 64, 16, 1025),
                                              (128, 64, 64, 1300)])
def test_paged_plans_of_few_waves_match_float64(gpu, D, H, page, longest):
    # enough (b,h) for the GPU: the plan's one to four waves per (b,h), not eight
    lens = [longest, 1, 63, 64, 65, 0, longest - 1, longest // 2] * 4
    B = len(lens)
    assert 1 <= capi.decode_num_splits(B * H, longest, D) <= 4
    c = workloads.paged_case(B, H, D, page, lens, seed=D + H, device=gpu)
    out = capi.decode_attention_paged(c["Qi"], c["K_pages"], c["V_pages"], c["sQ"],
                                      c["sK_pages"], c["sV_pages"], c["block_tables"],
                                      c["context_lens"], c["max_context"])
    torch.cuda.synchronize()
    for b in list(range(8)) + [B - 2]:
        o, n = out[b].float().cpu().numpy(), lens[b]
        if n == 0:
            assert np.all(o == 0)
            continue
        t = c["block_tables"][b, :-(-n // page)].long()
        flat = {k: c[k][t].transpose(0, 1).reshape(H, len(t) * page, -1)[:, :n]
                for k in ("K_pages", "V_pages", "sK_pages", "sV_pages")}
        ref = _ref(dict(Qi=c["Qi"][b:b + 1], sQ=c["sQ"].reshape(B, H)[b:b + 1],
                        Ki=flat["K_pages"][None], Vi=flat["V_pages"][None],
                        sK=flat["sK_pages"][None, ..., 0], sV=flat["sV_pages"][None, ..., 0]), n)
        assert_attn_close(o, ref[0], f"paged D{D} H{H} page{page} len{n}")
