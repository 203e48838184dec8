"""The MLP's few-token and 128 x 128-tile GEMMs at the edges of their tiles and splits.

Rows around the 32- and 64-row blocks of the streaming kernel and the 128-row tiles, K and N
off the 128 grid (the API asks for multiples of 16), K ranges that leave the last wave or split
short or empty, small weights on the skinny kernel (as stored: through transposed copies), the
widest row of the fused epilogue (32768 columns) and one past it, both weight layouts, bias,
scalar scales and the per-tensor output.  The integer sums are exact, so the codes are within
one of the oracle's and at most 2% of them differ (an fp32 epilogue in another order moves a
code only on a rounding tie), as in test_mlp_gpu.py.
"""
import numpy as np
import pytest
import torch

import int8k_capi as capi
import workloads
from oracle import int8_oracle as O
from oracle import oracle_c

pytestmark = pytest.mark.gpu

P = capi.MLP_WEIGHTS_PREPACKED
PT = capi.MLP_OUT_PER_TENSOR


def _check(T, dm, dff, gpu, bias=False, scalar=False):
    c = workloads.mlp_case(T, dm, dff, seed=T + dm + dff, device=gpu, gen_device="cpu")
    x = c["x"].reshape(T, dm)
    b = (torch.randn(dff, generator=torch.Generator().manual_seed(T)) * 0.5).to(gpu) if bias else None
    scales = (c["sx"], c["sW1"], c["sW2"])
    if scalar:
        scales = tuple(s.reshape(-1)[:1].clone() for s in scales)
    W1T, W2T = capi.transpose_int8_weights(c["W1"], c["W2"])
    n = [t.cpu().numpy() for t in (x, c["W1"], c["W2"], *scales)]
    for flags in (0, PT):
        ref, rsc = O.mlp_forward(*n, bias1=None if b is None else b.cpu().numpy(),
                                 per_token_out=flags == 0, gemm=oracle_c.gemm_i8_i32)
        for w1, w2, f in ((c["W1"], c["W2"], flags), (W1T, W2T, flags | P)):
            out, osc = capi.mlp_forward(x, w1, w2, *scales, bias1=b, flags=f)
            torch.cuda.synchronize()
            label = f"T{T} {dm}->{dff} flags {f}"
            d = np.abs(out.cpu().numpy().astype(np.int32) - ref.astype(np.int32))
            assert d.max() <= 1, f"{label}: off by {d.max()}"
            assert (d != 0).mean() <= 0.02, f"{label}: {(d != 0).mean()} differ"
            np.testing.assert_allclose(osc.cpu().numpy().reshape(-1), np.asarray(rsc).reshape(-1),
                                       rtol=2e-3, err_msg=label)


@pytest.mark.parametrize("T", [1, 31, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("dm,dff", [(400, 1040), (1296, 2064), (1552, 2064)])  # 3 MiB between
def test_stream_row_blocks(gpu, T, dm, dff):
    _check(T, dm, dff, gpu, bias=T % 2 == 1, scalar=T == 32)


@pytest.mark.parametrize("T,dm,dff", [
    (3, 16, 16), (5, 16, 4112), (2, 4112, 16), (1, 144, 128), (40, 2192, 784),
    (2, 48, 32768), (2, 48, 32784), (3, 6160, 64),
    (32, 528, 1024), (32, 256, 1040),        # weights of at most 3 MiB: up to 32 rows
])
def test_stream_edges(gpu, T, dm, dff):
    _check(T, dm, dff, gpu, bias=True)


@pytest.mark.parametrize("T,dm,dff", [
    (129, 1296, 2064), (256, 2064, 784), (257, 784, 4112), (333, 1040, 4112), (513, 528, 2192),
    (640, 2048, 1536), (130, 1040, 16400),
    (33, 16, 16), (100, 16, 4112), (64, 512, 1024), (128, 256, 1040), (300, 512, 1040),
    (33, 528, 1040), (128, 1040, 2064),  # weights of at most 3 MiB: from 33 rows
])
def test_mid_tiles_and_splits(gpu, T, dm, dff):
    _check(T, dm, dff, gpu, bias=T % 2 == 0)


@pytest.mark.parametrize("T,dm,dff", [
    # both GEMMs, packed; as stored through transposed copies above 128 rows, below 2^29
    # multiply-adds: the range's ends, GEMM2 alone (K = 1040 is off the kernel's grid), row tails
    (1, 512, 512), (33, 512, 1024), (128, 512, 512), (129, 512, 512), (257, 512, 1024),
    (1280, 512, 512), (2047, 512, 512), (2048, 512, 512), (511, 512, 2048), (200, 1024, 1024), (640, 512, 1024), (140, 1024, 96),
    (16, 1024, 3072), (64, 1024, 3072), (140, 640, 512),
])
def test_skinny_with_copies(gpu, T, dm, dff):
    _check(T, dm, dff, gpu, bias=T % 2 == 1)


def test_stream_unaligned_scales(gpu):
    # column scales and bias off the 16-byte grid are read one by one
    T, dm, dff = 17, 512, 1040
    c = workloads.mlp_case(T, dm, dff, seed=9, device=gpu, gen_device="cpu")
    x = c["x"].reshape(T, dm)
    b = torch.randn(dff + 1, generator=torch.Generator().manual_seed(2)).to(gpu)
    sh = [torch.cat([s.new_zeros(1), s])[1:] for s in (c["sW1"], c["sW2"])]
    for w in sh:
        assert w.data_ptr() % 16 != 0
    a = capi.mlp_forward(x, c["W1"], c["W2"], c["sx"], *sh, bias1=b[1:])
    e = capi.mlp_forward(x, c["W1"], c["W2"], c["sx"], c["sW1"], c["sW2"], bias1=b[1:].clone())
    torch.cuda.synchronize()
    assert torch.equal(a[0], e[0]) and torch.equal(a[1], e[1])
