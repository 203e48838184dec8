"""Row kernels at row lengths that do not fill their lanes: 16-byte chunk counts around the
powers of two, the per-lane instances (1, 2, 3, 4, 6, 8, 12, 16), where the last chunk is
repeated in the spare slots, and LayerNorm's switch to a block per row above 768 columns.
The quantizers are exact against the oracle; LayerNorm as in test_producer_gpu.py: one
storage ulp of y (its fp32 row sums differ from float64 by ~sqrt(cols) roundings, covered by
2^-17 relative for fp32)."""
import numpy as np
import pytest
import torch

import int8k_capi as capi
from oracle import int8_oracle as O

pytestmark = pytest.mark.gpu

_DT = {torch.float16: "f16", torch.bfloat16: "bf16", torch.float32: "f32"}
COLS = [8, 24, 80, 520, 768, 776, 1600, 2040, 2056, 2568, 4096, 5128, 6152, 8184, 8200]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("cols", COLS)
def test_quantize_rows(gpu, dtype, cols):
    x = (torch.randn(67, cols, generator=torch.Generator().manual_seed(cols)) * 3).to(dtype)
    x[5] = 0
    q, s = capi.quantize_per_token(x.to(gpu))
    torch.cuda.synchronize()
    rq, rs = O.quantize_per_token(x.float().numpy())
    np.testing.assert_array_equal(q.cpu().numpy(), rq)
    np.testing.assert_array_equal(s.cpu().numpy(), rs)


@pytest.mark.parametrize("cols,dtype", [(24, torch.float16), (512, torch.float16),
                                        (768, torch.float16), (100, torch.float32)])
@pytest.mark.parametrize("groups", [1, 4095, 4096, 4097, 16385, 32769])
def test_quantize_row_groups(gpu, cols, dtype, groups):
    # waves of one row group (as many rows as fill 64 lanes) up to 4 x 1024 waves, of up to
    # four groups beyond, some of them past the end
    chunks = cols * dtype.itemsize // 16
    per = 64 >> min(6, (chunks - 1).bit_length())
    rows = groups * per - (per > 1)
    x = (torch.randn(rows, cols, device=gpu, generator=torch.Generator(gpu).manual_seed(rows))
         * 3).to(dtype)
    q, s = capi.quantize_per_token(x)
    torch.cuda.synchronize()
    at = sorted({i for n in (0, rows // 4, rows // 2, rows - 33) for i in range(n, n + 33)
                 if 0 <= i < rows})
    rq, rs = O.quantize_per_token(x[at].float().cpu().numpy())
    np.testing.assert_array_equal(q[at].cpu().numpy(), rq)
    np.testing.assert_array_equal(s[at].cpu().numpy(), rs)
    # every row: codes times scale within half a step, on the GPU
    d = (q.float() * s.unsqueeze(-1) - x.float()).abs().amax(-1)
    assert bool((d <= s * (0.5 + 1e-4)).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("cols", COLS)
@pytest.mark.parametrize("rows,shift", [(67, 0), (1100, 0), (3, 1)])
def test_layernorm_rows(gpu, dtype, cols, rows, shift):
    # shift: gamma and beta off the 16-byte grid, read one by one
    g = torch.Generator().manual_seed(rows + cols)
    x = (torch.randn(rows, cols, generator=g) * 2 + 0.5).to(dtype)
    gamma, beta = torch.rand(cols + 1, generator=g) + 0.5, torch.rand(cols + 1, generator=g) - 0.5
    q, s, y = capi.layernorm_quantize_per_token(
        x.to(gpu), gamma.to(gpu)[shift:shift + cols], beta.to(gpu)[shift:shift + cols], 1e-5,
        want_y=True)
    torch.cuda.synchronize()
    n = min(rows, 67)
    rq, rs, ry = O.layernorm_quantize_per_token(
        x[-n:].float().numpy(), gamma[shift:shift + cols].numpy(),
        beta[shift:shift + cols].numpy(), 1e-5, _DT[dtype])
    ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 2.0 ** -17}[dtype]
    yd = np.abs(y[-n:].float().cpu().numpy() - ry)
    # where (x - mean) rstd gamma and beta (at most 0.5) cancel, y is small but its roundings
    # are those of terms below |y| + 1: 8 of them (mean, rstd, the products and the sum)
    cancel = 8 * 2.0 ** -24
    assert np.all(yd <= ulp * np.maximum(np.abs(ry), 2.0 ** -14) + cancel), yd.max()
    assert np.abs(q[-n:].cpu().numpy().astype(np.int32) - rq).max() <= 1
    np.testing.assert_allclose(s[-n:].cpu().numpy(), rs, rtol=1e-3)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("Dh", [24, 40, 72, 80, 96, 120])
def test_heads_and_cache_append(ext, gpu, dtype, Dh):
    B, S, H = 2, 37, 3
    g = torch.Generator().manual_seed(Dh)
    x = (torch.randn(B, S, 3 * H * Dh, generator=g) * 3).to(dtype)
    outs = ext.quantize_heads(x.to(gpu), H, 3)
    ref = O.quantize_heads(x.float().numpy(), H, 3)
    for p in range(3):
        np.testing.assert_array_equal(outs[2 * p].cpu().numpy(), ref[p][0])
        np.testing.assert_array_equal(outs[2 * p + 1].cpu().numpy(), ref[p][1])
    k, v = (torch.randn(B, H, 5, Dh, generator=g).to(dtype) for _ in range(2))
    K, V = (torch.full((B, H, 16, Dh), 7, dtype=torch.int8, device=gpu) for _ in range(2))
    sK, sV = (torch.full((B, H, 16), 7.0, device=gpu) for _ in range(2))
    ext.kv_cache_append(k.to(gpu), v.to(gpu), K, V, sK, sV, 9)
    torch.cuda.synchronize()
    for new, cache, sc in ((k, K, sK), (v, V, sV)):
        rq, rs = O.quantize_per_token(new.float().numpy())
        c, s = cache.cpu().numpy(), sc.cpu().numpy()
        np.testing.assert_array_equal(c[:, :, 9:14], rq)
        np.testing.assert_array_equal(s[:, :, 9:14], rs)
        assert (c[:, :, :9] == 7).all() and (c[:, :, 14:] == 7).all()
        assert (s[:, :, :9] == 7).all() and (s[:, :, 14:] == 7).all()
