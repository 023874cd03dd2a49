"""The C ABI without a GPU: libmkimage.so loads, exports every entry point include/mkimage.h declares, and its
host-only calls behave (no device work here)."""
import ctypes
import pathlib
import re

import mkimage
import mkref

ROOT = pathlib.Path(__file__).resolve().parents[1]


def declared():
    text = (ROOT / "include" / "mkimage.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mk_[a-z0-9_]+)\s*\(", text)) - {"mk_probe_fn"})


def test_library_exports_every_declared_entry_point():
    lib = ctypes.CDLL(str(mkimage.LIB_PATH))
    names = declared()
    assert len(names) > 40
    missing = [n for n in names if not hasattr(lib, n)]
    assert not missing, missing


def test_binding_covers_the_header():
    assert sorted(mkimage.EXPORTS) == declared()


def test_version_and_error_state():
    L = mkimage.lib()
    assert b"gfx950" in L.mk_version()
    # a host-side argument error, no device touched
    assert L.mk_gemm(None, None) == 1
    assert b"null" in L.mk_last_error()
    assert L.mk_engine_create(None, None) == 1


def test_tensor_key_matches_oracle():
    L = mkimage.lib()
    for seed, name in [(0, "img_in.weight"), (7, "transformer_blocks.59.attn.to_q.weight"), (2**63 + 5, "")]:
        assert L.mk_tensor_key(seed, name.encode()) == mkref.tensor_key(seed, name)


def test_bf16_rule_matches_oracle():
    import numpy as np

    x = np.random.default_rng(0).standard_normal(10000).astype(np.float32) * 1e3
    assert np.array_equal(mkimage.bf16_bits(x), mkref.bf16_bits(x))


def test_e4m3_codes_match_oracle():
    import numpy as np

    t = mkimage._e4m3_table()
    ref = mkref.e4m3_table()
    ok = ~np.isnan(ref)
    assert np.array_equal(t[ok], ref[ok])


def test_sigmas_match_oracle():
    import numpy as np

    for steps, tokens, terminal in [(40, 4096, 0.0), (1, 256, 0.0), (2, 256, 0.0), (30, 1024, 0.02), (7, 16384, 0.1),
                                    (1, 4096, 0.05)]:
        got = mkimage.sigmas(steps, tokens, terminal)
        want = mkref.sigmas(steps, tokens, terminal=terminal)
        assert np.array_equal(got, want), (steps, tokens, terminal)


def test_sigmas_fixed_shift_and_errors():
    import numpy as np

    # a fixed mu replaces the size-dependent line: the 2-step schedule is e^mu / (e^mu + 1) at t = 1/2
    s = mkimage.sigmas(2, 999, mu=1.5)
    assert s[0] == 1.0 and s[2] == 0.0
    assert abs(s[1] - np.exp(1.5) / (np.exp(1.5) + 1)) < 1e-7
    assert np.array_equal(mkimage.sigmas(5, 1, mu=0.7), mkimage.sigmas(5, 123456, mu=0.7))
    with __import__("pytest").raises(mkimage.MkError, match="max_seq"):
        mkimage.sigmas(4, 256, base_seq=100.0, max_seq=100.0)


def test_rope_table_is_the_oracle_table_bit_for_bit():
    # the engine uploads mk_rope_table's output; the oracle's table is pinned to the closed form in test_oracle.py
    import numpy as np

    for S, h, w in [(256, 64, 64), (7, 5, 3), (0, 4, 6), (512, 128, 128), (41, 1, 1)]:
        got = mkimage.rope_table(S, h, w)
        want = mkref.rope_table(S, h, w)
        assert got.view(np.uint32).tobytes() == want.view(np.uint32).tobytes(), (S, h, w)


def test_noise_restatement_is_pinned_by_the_standard():
    # [rand.predef]: the 10000th output of a default-constructed std::mt19937_64 (seed 5489)
    g = mkref.mt19937_64(5489)
    for _ in range(9999):
        next(g)
    assert next(g) == 9981545732273789042
    # moments of the polar method's draws
    z = mkref.noise(3, 20000)
    assert abs(z.mean()) < 0.03 and abs(z.std() - 1.0) < 0.03


def test_noise_matches_the_oracle_bit_for_bit():
    import numpy as np
    for seed, n in ((0, 1001), (1, 2), (42, 257), (2 ** 63 + 5, 64)):
        got = mkimage.noise(seed, n)
        want = mkref.noise(seed, n)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), seed
    # one draw is the first of a pair; two calls of one draw each are the same first value
    assert mkimage.noise(7, 1)[0] == mkimage.noise(7, 2)[0]


def test_vae_up_plan():
    # the 2x grid is written by the convolution where that measured faster than the pass of its own (256 compute units):
    # any width of whole tiles; else convolutions on 256 x 192 tiles in more than two rounds, or two nearly full ones
    def plan(h, w, c, cus=256):
        out = ctypes.c_uint32(7)
        mkimage.call("mk_vae_up_plan", h, w, c, cus, ctypes.byref(out))
        return out.value

    assert [plan(h, w, 384) for h, w in ((304, 208), (340, 224), (256, 256), (464, 260), (372, 310))] == [1] * 5
    # other tiles, two rounds of 402 to 452 tiles, a small level
    assert [plan(h, w, 384) for h, w in ((304, 216), (320, 208), (280, 180), (320, 176), (152, 104))] == [0] * 5
    assert [plan(h, w, 192) for h, w in ((608, 416), (456, 272), (576, 304), (288, 512))] == [1] * 4
    assert [plan(h, w, 192) for h, w in ((464, 288), (368, 360), (304, 240), (48, 48))] == [0] * 4
    # rounds are the device's: twice the image on twice the units, half of it on half
    assert plan(608, 208, 384, 512) == plan(304, 208, 384, 256) == plan(152, 208, 384, 128) == 1
    assert mkimage.lib().mk_vae_up_plan(304, 208, 100, 256, ctypes.byref(ctypes.c_uint32())) == 1


def _plan(rows, n, k, epi=0, w_dtype=mkimage.BF16, cus=256):
    g = mkimage.GemmArgs()
    g.a = g.w = g.c = g.gate = g.wscale = 4096  # (not read)
    g.M, g.N, g.K, g.lda, g.ldc, g.batch = rows, n, k, k, n, 1
    g.w_dtype, g.c_dtype, g.epilogue = w_dtype, mkimage.F32, epi
    out = (ctypes.c_uint32 * 3)()
    mkimage.call("mk_gemm_plan", ctypes.byref(g), 1, cus, out)
    return tuple(out)


def test_gemm_plan_splits():
    # below 1024 rows a tile's k steps are split while that is estimated faster, at most a workgroup a compute unit; never
    # for an epilogue the weight type has not
    assert _plan(77, 3072, 12288)[2] == 10 and _plan(320, 3072, 12288)[2] == 3
    assert _plan(1023, 256, 12288)[2] > 1 and _plan(1024, 256, 12288)[2] == 1
    assert _plan(1, 128, 832)[2] == 1 and _plan(1, 128, 896)[2] == 4  # 13 and 14 k steps
    assert _plan(1, 128, 576, w_dtype=mkimage.FP8)[2] == 1 and _plan(1, 128, 640, w_dtype=mkimage.FP8)[2] == 4
    assert _plan(512, 1280, 1280)[2] == 1
    for rows, n, k in ((1, 128, 12288), (300, 640, 12288), (900, 1024, 12288), (1023, 1920, 8192)):
        tiles = -(-rows // 128) * (n // 128)
        for wdt in (mkimage.BF16, mkimage.FP8, mkimage.F16):
            splits = _plan(rows, n, k, w_dtype=wdt)[2]
            assert splits == 1 or (splits * tiles <= 256 and splits * rows * n * 4 <= 32 << 20)
    for epi in (mkimage.EPI_GELU_TANH, mkimage.EPI_SILU):
        assert _plan(77, 3072, 12288, epi)[2] > 1
        assert _plan(77, 3072, 12288, epi, mkimage.F16)[2] == 1
