"""The MFMA attention at the edges of its query tiles (32), key blocks (32), rounds (128 keys) and
head pairs, through a block: causal behind an existing context, and scores whose row max keeps
rising over the keys.  Fewer queries than a tile take the scalar kernel, here with long contexts
and caches and with value rows of infinities and NaN."""
import numpy as np
import pytest

from test_gpu_minicpm4 import _dev, cfg_dict, orc_cfg, rand_layer, to_orc

pytestmark = pytest.mark.gpu


# nh / nkv: pairs of heads share a kv head (4 / 2 with a full device, 16 / 2), or none does
# (3 / 3); 16 heads x 33 tiles and more run two heads per workgroup
@pytest.mark.parametrize("M,pos,nh,nkv,hd", [(2, 127, 4, 2, 128), (31, 98, 4, 2, 64), (32, 0, 3, 3, 128), (33, 0, 4, 2, 64),
                                             (64, 64, 4, 2, 128), (65, 63, 4, 2, 128), (96, 33, 3, 3, 64),
                                             (127, 1, 4, 2, 128), (129, 0, 16, 2, 64), (2, 2000, 4, 2, 128),
                                             (1025, 0, 16, 2, 64), (1056, 0, 16, 2, 128), (1030, 7, 12, 12, 64)])
@pytest.mark.parametrize("rising", [False, True])
def test_block_at_tile_edges(vxm_ctx, orc, M, pos, nh, nkv, hd, rising):
    import vxm

    rng = np.random.default_rng(M + pos + nh + hd)
    H, F, cap = 256, 256, (M + pos + 63) // 64 * 64
    lw = rand_layer(orc, rng, H, nh, nkv, hd, F)
    c = cfg_dict(H, 1, nh, nkv, hd, F)
    # rising: keys that grow with their position, so the running max rises again and again
    grow = np.linspace(0.1, 12.0, cap)[None, :, None] if rising else 1.0
    k = orc.fp32_to_fp16_bits(orc.bf16_round((rng.normal(0, 1, (nkv, cap, hd)) * grow).astype(np.float32)))
    v = orc.fp32_to_fp16_bits(orc.bf16_round(rng.normal(0, 1, (nkv, cap, hd)).astype(np.float32)))
    k[:, pos:] = 0
    v[:, pos:] = 0
    x = rng.normal(0, 1, (M, H)).astype(np.float32)
    model = vxm.MiniCPM4(vxm_ctx, c, [lw])
    kv = vxm.KVCache(vxm_ctx, 1, nkv, hd, cap)
    kv.upload(0, k, v)
    xd = _dev(x)
    model.block(kv, 0, xd, pos)
    vxm_ctx.sync()
    kc, vc = k.reshape(-1).copy(), v.reshape(-1).copy()
    ref = orc.minicpm4_block(orc_cfg(orc, c), to_orc(orc, lw), x, kc, vc, cap, pos, 0)
    # the block sensitivity bar: one BF16 ulp on one element of a block's input moves the oracle's own
    # output by up to 4e-3 (relative L2), as another order of the fp32 sums may
    y = xd.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(y - ref) <= 5e-3 * np.linalg.norm(ref), np.linalg.norm(y - ref) / np.linalg.norm(ref)
    assert np.all(np.abs(y - ref) <= 2.0 ** -6 * np.abs(ref).max(axis=1, keepdims=True))
    kv.free()
    model.free()


def test_block_noncausal_tile_edges(vxm_ctx, orc):
    """Non-causal spans that end inside a key block, a round and a tile."""
    import vxm

    rng = np.random.default_rng(5)
    H, nh, nkv, hd, F = 256, 4, 2, 64, 256
    lw = rand_layer(orc, rng, H, nh, nkv, hd, F)
    c = cfg_dict(H, 1, nh, nkv, hd, F)
    model = vxm.MiniCPM4(vxm_ctx, c, [lw])
    for M in (130, 161, 257):
        x = rng.normal(0, 1, (M, H)).astype(np.float32)
        xd = _dev(x)
        model.block(None, 0, xd, 0, no_causal=1)
        vxm_ctx.sync()
        ref = orc.minicpm4_block(orc_cfg(orc, c), to_orc(orc, lw), x, None, None, 0, 0, 1)
        y = xd.cpu().numpy().astype(np.float64)
        assert np.linalg.norm(y - ref) <= 5e-3 * np.linalg.norm(ref), M
    model.free()


@pytest.mark.parametrize("M,pos,hd", [(2, 127, 128), (5, 300, 64), (31, 98, 128), (31, 1000, 64)])
def test_overflowing_value_row_reaches_no_earlier_token(vxm_ctx, orc, M, pos, hd):
    """The last token's value row holds infinities (past f16); the tokens before it do not see it."""
    import vxm

    rng = np.random.default_rng(M + pos)
    H, nh, nkv, F, cap = 256, 4, 2, 256, (M + pos + 63) // 64 * 64
    lw = rand_layer(orc, rng, H, nh, nkv, hd, F)
    wv = rng.normal(0, 0.02, (nkv * hd, H)).astype(np.float32)
    wv[:, 0] = 0
    wv[::hd] = 0
    wv[::hd, 0] = 1e6            # dim 0 of every value head: 1e6 x channel 0 of the normalised row
    lw["v_proj"] = orc.quantize_rows(wv, orc.QUANT_REF)
    k = orc.fp32_to_fp16_bits(orc.bf16_round(rng.normal(0, 1, (nkv, cap, hd)).astype(np.float32)))
    v = orc.fp32_to_fp16_bits(orc.bf16_round(rng.normal(0, 1, (nkv, cap, hd)).astype(np.float32)))
    x = rng.normal(0, 1, (M, H)).astype(np.float32)
    x[:, 0] = 0                  # no other token has channel 0
    model = vxm.MiniCPM4(vxm_ctx, cfg_dict(H, 1, nh, nkv, hd, F), [lw])
    kv = vxm.KVCache(vxm_ctx, 1, nkv, hd, cap)
    ys = []
    for big in (0.0, 5.0):
        kv.upload(0, k, v)
        x[-1, 0] = big
        xd = _dev(x)
        model.block(kv, 0, xd, pos)
        vxm_ctx.sync()
        ys.append(xd.cpu().numpy())
    assert np.isfinite(ys[0]).all()
    assert np.isinf(kv.download(0)[1].view(np.float16)[:, pos + M - 1, 0]).all()
    assert np.array_equal(ys[0][:-1], ys[1][:-1])
    kv.free()
    model.free()


# past 40624 rows (64 dims) the scalar kernel's score buffer holds no more than the call's own
# keys; a call with more of them takes the MFMA kernel
@pytest.mark.parametrize("M,pos,cap", [(5, 300, 20000), (1, 98, 40624), (31, 98, 40624), (31, 98, 40625), (2, 127, 45000),
                                       (31, 1000, 45000), (5, 40800, 45000)])
def test_few_queries_in_a_long_cache(vxm_ctx, orc, M, pos, cap):
    import vxm

    rng = np.random.default_rng(M + pos + cap)
    H, nh, nkv, hd, F = 256, 4, 2, 64, 256
    lw = rand_layer(orc, rng, H, nh, nkv, hd, F)
    c = cfg_dict(H, 1, nh, nkv, hd, F)
    k = orc.fp32_to_fp16_bits(orc.bf16_round(rng.normal(0, 1, (nkv, cap, hd)).astype(np.float32)))
    v = orc.fp32_to_fp16_bits(orc.bf16_round(rng.normal(0, 1, (nkv, cap, hd)).astype(np.float32)))
    x = rng.normal(0, 1, (M, H)).astype(np.float32)
    model = vxm.MiniCPM4(vxm_ctx, c, [lw])
    kv = vxm.KVCache(vxm_ctx, 1, nkv, hd, cap)
    kv.upload(0, k, v)
    xd = _dev(x)
    model.block(kv, 0, xd, pos)
    vxm_ctx.sync()
    y = xd.cpu().numpy().astype(np.float64)
    ref = orc.minicpm4_block(orc_cfg(orc, c), to_orc(orc, lw), x, k.reshape(-1).copy(), v.reshape(-1).copy(), cap, pos, 0)
    assert np.linalg.norm(y - ref) <= 5e-3 * np.linalg.norm(ref)
    kv.free()
    model.free()


def test_nan_output_quantizes_as_by_itself(vxm_ctx, orc):
    """Under the reference's rounding rule a NaN value quantizes to 0 in k_quantize_q8_0; so it does
    where the attention of few queries writes the Q8_0 rows: a value dim that holds a NaN gives what
    one of zeros gives."""
    import vxm

    rng = np.random.default_rng(17)
    H, nh, nkv, hd, F, cap, M, pos, dim = 256, 4, 2, 128, 256, 128, 5, 60, 37
    lw = rand_layer(orc, rng, H, nh, nkv, hd, F)
    wv = rng.normal(0, 0.02, (nkv * hd, H)).astype(np.float32)
    wv[dim] = 0
    lw["v_proj"] = orc.quantize_rows(wv, orc.QUANT_REF)
    k = orc.fp32_to_fp16_bits(orc.bf16_round(rng.normal(0, 1, (nkv, cap, hd)).astype(np.float32)))
    v = orc.fp32_to_fp16_bits(orc.bf16_round(rng.normal(0, 1, (nkv, cap, hd)).astype(np.float32)))
    v[0, :, dim] = 0
    x = rng.normal(0, 1, (M, H)).astype(np.float32)
    model = vxm.MiniCPM4(vxm_ctx, cfg_dict(H, 1, nh, nkv, hd, F), [lw])
    kv = vxm.KVCache(vxm_ctx, 1, nkv, hd, cap)
    ys = []
    try:
        vxm_ctx.set_quant_variant(vxm.QUANT_REF)
        for bits in (0, 0x7E00):
            v[0, 3, dim] = bits
            kv.upload(0, k, v)
            xd = _dev(x)
            model.block(kv, 0, xd, pos)
            vxm_ctx.sync()
            ys.append(xd.cpu().numpy())
    finally:
        vxm_ctx.set_quant_variant(vxm.QUANT_X86)
    assert np.isfinite(ys[0]).all() and np.array_equal(ys[0], ys[1])
    kv.free()
    model.free()
