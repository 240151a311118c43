"""Short prompts (2 to 128 tokens) against the oracle: the small-M GEMM past one row tile and
with three wave groups, the rope kernel over K-split slices, and the per-token attention with
its Q8_0 output, at the sizes where their tiles, slices and vector loads end."""
import numpy as np
import pytest

from test_gpu_minicpm4 import _dev, cfg_dict, orc_cfg, rand_layer, to_orc

pytestmark = pytest.mark.gpu


# K = 6144 over 8 splits: three stages per split, three wave groups.  65 to 128 rows: two row
# tiles (of 48 or 64 rows, the last one ragged), K splits (the tile GEMM would split K there).
# 64 x 256 at 65 rows and 2560 x 2048 at 77 go to the tile GEMM: the tile's plan is unsplit, and
# the small-M grid more than one round.
@pytest.mark.parametrize("N,K,M", [(64, 6144, 1), (64, 6144, 16), (2048, 6144, 17), (2048, 6144, 32), (2048, 6144, 33),
                                   (64, 256, 65), (2048, 2048, 65), (2048, 2048, 96), (2048, 2048, 97),
                                   (1024, 4096, 127), (512, 2048, 128), (2048, 6144, 128), (2560, 2048, 77),
                                   (64, 1536, 65), (192, 4864, 77)])
def test_small_gemm_row_tiles_and_wave_groups(vxm_ctx, orc, N, K, M):
    import vxm

    kernel = vxm.host_mul_mat_plan(N, K, M, vxm.PATH_MFMA, rows=vxm.ROWS_Q8)[0]
    assert kernel == ("tile" if (N, K, M) in ((64, 256, 65), (2560, 2048, 77)) else "small")
    rng = np.random.default_rng(N + 3 * K + 7 * M)
    x = rng.normal(0, 1, (M, K)).astype(np.float32)
    wq = orc.quantize_rows(rng.normal(0, 0.02, (N, K)).astype(np.float32), orc.QUANT_REF)
    w = vxm_ctx.upload_q8_0(wq, N, K)
    xq, xd = vxm_ctx.quantize_q8_0(_dev(x), 1)
    xq_ref = orc.quantize_rows(x, 1)
    ref = orc.mul_mat_f64(wq, xq_ref, N, K, M)
    try:
        vxm_ctx.set_path(vxm.PATH_MFMA)
        y, dots = vxm_ctx.mul_mat_q8(w, xq, xd), vxm_ctx.block_dots(w, xq, xd)
        vxm_ctx.sync()
        y = y.cpu().numpy()
        assert np.array_equal(dots.cpu().numpy(), orc.block_dots(wq, xq_ref, N, K, M))
    finally:
        vxm_ctx.set_path(vxm.PATH_AUTO)
    err = np.abs(y - ref)
    assert np.all(err <= 1e-4 + 1e-3 * np.abs(ref)), err.max()
    w.free()


# head sizes: 64 and 128 (Q8_0 blocks fused, 16-byte key rows), 96 (a ragged last group of key
# loads), 48 (16-byte rows, Q8_0 in a launch of its own), 20 (neither)
@pytest.mark.parametrize("M,pos,nh,hd", [(2, 0, 4, 128), (9, 31, 4, 64), (31, 0, 4, 128), (24, 300, 4, 128),
                                         (65, 0, 4, 128), (100, 300, 4, 128), (128, 0, 4, 64), (7, 5, 4, 96),
                                         (7, 40, 8, 48), (7, 40, 8, 20)])
def test_short_prompt_block(vxm_ctx, orc, M, pos, nh, hd):
    import vxm

    rng = np.random.default_rng(11 * M + pos + hd)
    H, nkv, F, cap = 2048, 2, 512, 512
    lw = rand_layer(orc, rng, H, nh, nkv, hd, F)
    c = cfg_dict(H, 1, nh, nkv, hd, F)
    prior = [orc.fp32_to_fp16_bits(orc.bf16_round(rng.normal(0, 1, (nkv, cap, hd)).astype(np.float32))) for _ in "kv"]
    for p in prior:
        p[:, pos:] = 0
    x = rng.normal(0, 1, (M, H)).astype(np.float32)
    model = vxm.MiniCPM4(vxm_ctx, c, [lw])
    kv = vxm.KVCache(vxm_ctx, 1, nkv, hd, cap)
    kv.upload(0, *prior)
    xd = _dev(x)
    model.block(kv, 0, xd, pos)
    vxm_ctx.sync()
    kc, vc = (p.reshape(-1).copy() for p in prior)
    ref = orc.minicpm4_block(orc_cfg(orc, c), to_orc(orc, lw), x, kc, vc, cap, pos, 0)
    # full-width rows: the block sensitivity bar.  One BF16 ulp on one input element moves the
    # oracle's own block output by up to 4e-3 (relative L2; every activation is re-quantized to 8
    # bits), so another order of the fp32 sums may do as much.
    y = xd.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(y - ref) <= 5e-3 * np.linalg.norm(ref), np.linalg.norm(y - ref) / np.linalg.norm(ref)
    assert np.all(np.abs(y - ref) <= 2.0 ** -6 * np.abs(ref).max(axis=1, keepdims=True))
    for got, want in zip(kv.download(0), (kc, vc)):
        g, r = orc.fp16_bits_to_fp32(got.reshape(-1)), orc.fp16_bits_to_fp32(want)
        assert np.abs(g - r).max() <= 2 ** -7 * np.abs(r).max()
    kv.free()
    model.free()
