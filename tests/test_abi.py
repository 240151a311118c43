"""CPU tests of the C ABI library: it loads, exports every declared symbol,
and its host-only helpers agree with the oracle.  No device work here."""
import os

import numpy as np

from conftest import GOLDEN, ROOT


def test_library_exports_every_header_symbol():
    import vxm

    names = vxm.header_functions()
    assert len(names) >= 20
    L = vxm.lib()
    missing = [n for n in names if not hasattr(L, n)]
    assert not missing, missing
    # the Python mirror binds every declared function with a signature
    assert set(names) <= set(vxm._SIGS), set(names) - set(vxm._SIGS)


def test_open_without_device_fails_cleanly():
    import torch
    import vxm

    if torch.cuda.is_available():
        return  # on a GPU host opening succeeds; covered by the gpu tests
    try:
        vxm.Context(0)
    except vxm.VxmError as e:
        assert e.code in (4, 5)
    else:
        raise AssertionError("vxm_open succeeded without a device")


def test_host_quantize_matches_oracle(orc):
    import vxm

    rng = np.random.default_rng(7)
    x = rng.normal(0, 0.02, (33, 256)).astype(np.float32)
    x[3, 32:64] = 0.0
    assert np.array_equal(vxm.host_quantize_q8_0(x), orc.quantize_rows(x, orc.QUANT_REF))


def test_host_quantize_golden():
    import vxm

    g = np.load(os.path.join(GOLDEN, "q8_cases.npz"))
    for i in range(6):
        if f"c{i}_w" in g:
            assert np.array_equal(vxm.host_quantize_q8_0(g[f"c{i}_w"]), g[f"c{i}_wq"])


def test_host_randn_is_seeded_sliceable_and_normal():
    import vxm

    a = vxm.host_randn(0, 100_001, 0.0, 1.0)
    b = vxm.host_randn(0, 100_001, 0.0, 1.0)
    assert np.array_equal(a, b)
    # any slice is reproducible on its own
    assert np.array_equal(vxm.host_randn(0, 1000, 0.0, 1.0, offset=4321), a[4321:5321])
    assert np.array_equal(vxm.host_randn(0, 7, 0.0, 1.0, offset=99_990), a[99_990:99_997])
    assert abs(a.mean()) < 0.02 and abs(a.std() - 1.0) < 0.02
    c = vxm.host_randn(1, 100_000, 0.0, 0.02)
    assert abs(c.std() - 0.02) < 0.001
    assert not np.array_equal(c[:10] / 0.02, a[:10])
    # first values are the Box-Muller pair of SplitMix64 outputs 1 and 2
    G = 0x9E3779B97F4A7C15
    M64 = (1 << 64) - 1

    def mix(z):
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
        return z ^ (z >> 31)

    u1 = ((mix(G) >> 11) + 1) * 2.0 ** -53
    u2 = (mix(2 * G & M64) >> 11) * 2.0 ** -53
    r = np.sqrt(-2 * np.log(u1))
    assert a[0] == np.float32(r * np.cos(2 * np.pi * u2))
    assert a[1] == np.float32(r * np.sin(2 * np.pi * u2))


def test_graft_entry_has_build_and_smoke():
    import importlib.util

    spec = importlib.util.spec_from_file_location("ge", os.path.join(ROOT, "__graft_entry__.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    assert callable(m.build) and callable(m.smoke)


def test_mul_mat_plans():
    """The kernel and K splits of the dispatch at the lines between its kernels."""
    import vxm

    plan = vxm.host_mul_mat_plan
    for n, k, m, rows, want in [
            (6144, 2048, 7, 0, ("gemv", 1)), (6144, 2048, 8, 0, ("small", 4)), (12288, 2048, 16, 0, ("small", 2)),
            # above one row tile: the tile GEMM where it needs no K split
            (12288, 2048, 17, 0, ("tile", 1)), (2048, 2048, 17, 0, ("small", 8)), (2048, 2048, 64, 0, ("small", 8)),
            (2048, 2048, 65, 0, ("small", 4)), (2048, 2048, 128, 0, ("small", 4)), (2048, 2048, 129, 0, ("tile", 2)),
            (2560, 2048, 64, 0, ("small", 8)), (2560, 2048, 65, 0, ("tile", 3)),
            (2048, 2080, 100, 0, ("staged", 4)), (96, 2048, 16, 0, ("tile", 4)),
            # fp32 rows
            (6144, 2048, 1, 1, ("gemv_f32", 1)), (6144, 2048, 2, 1, ("gemv_f32", 1)), (6144, 2048, 3, 1, ("gemv", 1)),
            (1024, 1024, 5, 1, ("gemv_f32", 1)), (1024, 1024, 6, 1, ("gemv", 1)),
            (8192, 1024, 5, 1, ("gemv_f32", 1)), (12288, 1024, 4, 1, ("gemv", 1)),
            (5, 6144, 2, 1, ("gemv_f32", 1)), (5, 6144, 3, 1, ("gemv", 1)), (5, 9216, 1, 1, ("gemv_f32", 1)),
            (5, 9248, 1, 1, ("gemv", 1)), (512, 40960, 1, 1, ("gemv", 1)), (16384, 256, 1, 1, ("gemv_f32", 1)),
            (16388, 256, 1, 1, ("gemv", 1)), (3072, 6144, 1, 1, ("gemv_f32", 1)), (4096, 6144, 1, 1, ("gemv", 1)),
            (32000, 4096, 1, 1, ("gemv", 1)), (4096, 11008, 1, 1, ("gemv", 1)), (73448, 2048, 1, 1, ("gemv", 1)),
            (6144, 2048, 16, 1, ("small_f32", 4)), (6144, 2048, 32, 1, ("small", 4)), (12288, 2048, 8, 1, ("small", 2)),
            (2048, 2048, 32, 1, ("small_f32", 8)), (2048, 2048, 33, 1, ("small", 8)),
            # whose stages are not too many in a row
            (512, 5632, 16, 1, ("small_f32", 8)), (512, 11008, 16, 1, ("small", 8)), (1024, 8192, 17, 1, ("small", 8)),
            # short K unsplit by the tile GEMM: while the launches cost less than its stages
            (2048, 256, 24, 0, ("small", 1)), (2048, 256, 49, 0, ("tile", 1)), (2048, 512, 24, 0, ("tile", 1)),
            (1024, 1024, 48, 0, ("small", 4)), (1024, 1024, 49, 0, ("tile", 1)),
            # two row tiles, by the stages in a row
            (2048, 4096, 128, 0, ("small", 4)), (2048, 5120, 77, 0, ("small", 4)), (2048, 5120, 100, 0, ("tile", 4)),
            (2048, 11008, 77, 0, ("tile", 4)),
            # a block's products, whose slices the next kernel adds
            (3072, 1024, 48, 2, ("small", 4)), (8192, 1024, 24, 2, ("small", 2)), (8192, 768, 48, 2, ("small", 2)),
            (8192, 768, 49, 2, ("tile", 1)), (12288, 2048, 24, 2, ("tile", 1)), (2048, 6144, 77, 2, ("small", 4)),
            (2560, 2048, 128, 2, ("small", 4)), (2560, 4096, 96, 2, ("small", 4)), (2560, 4096, 97, 2, ("tile", 3)),
            (2048, 11008, 77, 2, ("tile", 4)), (4096, 11008, 128, 2, ("tile", 2)),
            # a block's gate/up with SwiGLU in the epilogue; past 32-bit offsets the small-M GEMM up to one
            # row tile of its waves, above it refused as every tiled product of that size
            (12288, 2048, 32, 3, ("small", 1)), (12288, 2048, 33, 3, ("tile", 1)), (4096, 512, 48, 3, ("small", 1)),
            (4096, 512, 49, 3, ("tile", 1)), (1048512, 2048, 33, 3, ("small", 1)), (1048512, 2048, 64, 3, ("small", 1)),
            (1048512, 2048, 65, 3, ("none", 1)), (1048512, 2048, 128, 3, ("none", 1)),
            # two row tiles in three wave groups quantize in a launch of their own
            (1344, 6144, 16, 1, ("small_f32", 8)), (1344, 6144, 17, 1, ("small", 8)), (64, 768, 20, 1, ("tile", 1))]:
        assert plan(n, k, m, rows=rows) == want, (n, k, m, rows, plan(n, k, m, rows=rows))
    for path, want in ((vxm.PATH_GEMV, "gemv"), (vxm.PATH_MFMA, "small"), (vxm.PATH_MFMA_TILED, "tile")):
        assert plan(2048, 2048, 16, path, rows=vxm.ROWS_Q8)[0] == want


def test_mul_mat_plan_takes_operands_up_to_2_gib():
    """Up to 64 rows every weight below 2 GiB of quants runs: the small-M GEMM takes those that
    the tile GEMM, which addresses whole tiles past the last row, refuses."""
    import vxm

    for k in (256, 2048, 6144):
        n = ((1 << 31) // k - 1) // 64 * 64
        assert n * k < 1 << 31 and (n + 128) * k >= 1 << 31
        for m in (8, 16, 17, 24, 33, 64):
            assert vxm.host_mul_mat_plan(n, k, m)[0] == "small", (n, k, m)
        assert vxm.host_mul_mat_plan(n, k, 65)[0] == "none"
        assert vxm.host_mul_mat_plan(n - 192, k, 17)[0] != "none"
