"""The GEMV that quantizes its fp32 rows itself equals quantization and GEMV in launches of their
own bit for bit: every K that has a chunked kernel, the generic one, ragged row counts, the largest
row count it takes, both quantizers, zero and non-finite blocks, and an output over the input."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _host(ctx, t):
    ctx.sync()   # the library works on its own stream
    return t.cpu().numpy()


def _rows(rng, M, K, wild):
    """Rows with a zero block; wild: infinities, NaN and a block whose scale overflows fp16 in the
    last row's last blocks (everything that they reach stops being comparable by value)."""
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    x[0, :32] = 0.0
    if wild:
        x[-1, -1] = 3e38
        if K >= 96:
            x[-1, -40], x[-1, -70] = np.inf, np.nan
    return x


def _same(a, b, wild):
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert wild or np.isfinite(a).all()
    assert np.isfinite(a[:-1]).all()


# the last three are past the fused kernel's range
_TWO_LAUNCHES = [(3, 6144, 5), (7, 3072, 5), (5, 9248, 1)]


@pytest.mark.parametrize("N,K,M", [(64, 1024, 1), (1001, 1024, 5), (512, 2048, 1), (2051, 2048, 3), (2048, 4096, 2),
                                   (1023, 6144, 1), (2048, 512, 5), (1024, 64, 4), (5, 32, 1), (7, 6144, 2),
                                   (9, 4096, 3), (7, 3072, 4), (5, 9216, 1)] + _TWO_LAUNCHES)
@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("wild", [False, True])
def test_fused_gemv_equals_two_launches(vxm_ctx, orc, N, K, M, variant, wild):
    import torch
    import vxm

    assert vxm.host_mul_mat_plan(N, K, M)[0] == ("gemv" if (N, K, M) in _TWO_LAUNCHES else "gemv_f32")
    rng = np.random.default_rng(N + K + M)
    x = _rows(rng, M, K, wild)
    w = vxm_ctx.upload_q8_0(orc.quantize_rows(rng.normal(0, 0.02, (N, K)).astype(np.float32), orc.QUANT_REF), N, K)
    xd = torch.from_numpy(x).to("cuda:0")
    torch.cuda.synchronize()
    vxm_ctx.set_quant_variant(variant)
    try:
        y = _host(vxm_ctx, vxm_ctx.mul_mat(w, xd))
    finally:
        vxm_ctx.set_quant_variant(1)
    ref = _host(vxm_ctx, vxm_ctx.mul_mat_q8(w, *vxm_ctx.quantize_q8_0(xd, variant)))
    _same(y, ref, wild)
    w.free()


def test_output_over_the_input(vxm_ctx, orc):
    """y over x: no workgroup may read a row that another has overwritten."""
    import torch

    rng = np.random.default_rng(3)
    n = 2048
    w = vxm_ctx.upload_q8_0(orc.quantize_rows(rng.normal(0, 0.02, (n, n)).astype(np.float32), orc.QUANT_REF), n, n)
    x = torch.from_numpy(rng.normal(0, 1, (2, n)).astype(np.float32)).to("cuda:0")
    torch.cuda.synchronize()
    for rows in (1, 2):
        ref = _host(vxm_ctx, vxm_ctx.mul_mat_q8(w, *vxm_ctx.quantize_q8_0(x[:rows], 1)))
        y = x[:rows].clone()
        torch.cuda.synchronize()
        assert np.array_equal(_host(vxm_ctx, vxm_ctx.mul_mat(w, y, y)), ref)
    w.free()


@pytest.mark.parametrize("N,K,M", [(64, 256, 8), (2048, 6144, 16), (2048, 2048, 17), (1024, 4096, 31), (512, 2048, 32),
                                   (6144, 2048, 9), (64, 512, 10), (512, 5632, 13), (1024, 6144, 24)])
@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("wild", [False, True])
def test_fused_small_gemm_equals_three_launches(vxm_ctx, orc, N, K, M, variant, wild):
    """The small-M GEMM's own quantization (one row tile with one to three wave groups, several
    stages in a row, two row tiles; split and unsplit K) gives the bits of the separate launches.
    Two row tiles in three wave groups (the last shape) quantize in one."""
    import torch
    import vxm

    assert vxm.host_mul_mat_plan(N, K, M)[0] == ("small" if (K, M) == (6144, 24) else "small_f32")

    rng = np.random.default_rng(2 * N + K + M)
    x = _rows(rng, M, K, wild)
    w = vxm_ctx.upload_q8_0(orc.quantize_rows(rng.normal(0, 0.02, (N, K)).astype(np.float32), orc.QUANT_REF), N, K)
    xd = torch.from_numpy(x).to("cuda:0")
    torch.cuda.synchronize()
    vxm_ctx.set_quant_variant(variant)
    try:
        y = _host(vxm_ctx, vxm_ctx.mul_mat(w, xd))
    finally:
        vxm_ctx.set_quant_variant(1)
    ref = _host(vxm_ctx, vxm_ctx.mul_mat_q8(w, *vxm_ctx.quantize_q8_0(xd, variant)))
    _same(y, ref, wild)
    if N <= K:   # over the input: the same bits
        buf = xd.clone()
        torch.cuda.synchronize()
        vxm_ctx.set_quant_variant(variant)
        try:
            over = _host(vxm_ctx, vxm_ctx.mul_mat(w, buf, buf.view(-1)[:M * N].view(M, N)))
        finally:
            vxm_ctx.set_quant_variant(1)
        _same(over, ref, wild)
    w.free()
