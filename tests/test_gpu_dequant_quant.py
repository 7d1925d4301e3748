"""GPU parity: bulk dequantizers bit-exact with the oracle (which is pinned to
the reference's known answers), quantizers bit-exact with the reference's own
quantizer output (golden vectors) and with the oracle."""

from __future__ import annotations

from pathlib import Path

import numpy as np
import pytest
import torch

from gpu_helpers import announce, to_dev, to_np
from oracle import fp4 as ofp4

pytestmark = pytest.mark.gpu

GOLD = Path(__file__).resolve().parent / "golden" / "quantize_fp4_vectors.npz"


def _word(codes):
    w = 0
    for i, c in enumerate(codes):
        w |= (c & 0xF) << (4 * i)
    return w


def test_fp4_dequant_all_codes_all_fp16_scales():
    import mmfp4
    bits = np.arange(0x10000, dtype=np.uint32).astype(np.uint16)
    scales = bits.view(np.float16)          # includes inf / nan / subnormals
    n = scales.shape[0]
    packed = np.tile(np.array([[_word(range(8))], [_word(range(8, 16))]], np.uint32), (1, n))
    announce("fp4 dequant exhaustive 16 codes x 65536 scales")
    out = to_np(mmfp4.dequant_fp4(to_dev(packed), to_dev(scales.reshape(1, n)), 16, n, 16))
    ref = ofp4.dequant_fp4(packed, scales.reshape(1, n), 16)
    assert np.array_equal(out.view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("K,N,g", [(128, 64, 32), (1024, 520, 128), (4096, 4096, 128)])
def test_fp4_dequant_random(rng, K, N, g):
    import mmfp4
    packed = rng.integers(0, 2**32, (K // 8, N), dtype=np.uint64).astype(np.uint32)
    scales = rng.normal(0, 0.01, (K // g, N)).astype(np.float16)
    scales.reshape(-1)[:7] = [0.0, -0.0, 6e-8, 1e-5, 60000.0, np.inf, np.nan]
    announce(f"fp4 dequant random K={K} N={N} g={g}")
    out = to_np(mmfp4.dequant_fp4(to_dev(packed), to_dev(scales), K, N, g))
    ref = ofp4.dequant_fp4(packed, scales, g)
    assert np.array_equal(out.view(np.uint16), ref.view(np.uint16))


def test_u4_dequant_exhaustive_and_random(rng):
    import mmfp4
    # every q (column of 16 rows) x zero points x scales
    zs = np.concatenate([np.arange(-3, 19), rng.uniform(-3, 18, 42), [200.0, -300.0]])
    ss = np.concatenate([rng.uniform(1e-4, 4, 30), [0.0, 65504.0, np.inf, np.nan]])
    zz, sc = np.meshgrid(zs.astype(np.float16), ss.astype(np.float16))
    n = zz.size
    packed = np.tile(np.array([[_word(range(8))], [_word(range(8, 16))]], np.uint32), (1, n))
    announce(f"u4 dequant exhaustive n={n}")
    out = to_np(mmfp4.dequant_int4(to_dev(packed), to_dev(sc.reshape(1, n)),
                                   to_dev(zz.reshape(1, n)), 16, n, 16))
    ref = ofp4.dequant_u4(packed, sc.reshape(1, n), zz.reshape(1, n), 16)
    assert np.array_equal(out.view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("name", ["w_normal_f16", "w_crafted_f32", "w_crafted_f16",
                                  "w_normal_f32_g32"])
def test_quantize_fp4_matches_reference_vectors(name):
    import mmfp4
    d = np.load(GOLD)
    w, g = d[f"{name}__w"], int(d[f"{name}__g"])
    announce(f"quantize_fp4 golden {name}")
    packed, scales = mmfp4.quantize_fp4(to_dev(w), group_size=g)
    assert np.array_equal(to_np(packed).view(np.uint32), d[f"{name}__packed"])
    assert np.array_equal(to_np(scales).view(np.uint16), d[f"{name}__scales"].view(np.uint16))


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_quantize_fp4_random_vs_oracle(rng, dtype):
    import mmfp4
    w = rng.normal(0, 0.02, (384, 1024)).astype(dtype)
    announce(f"quantize_fp4 random {dtype.__name__}")
    packed, scales = mmfp4.quantize_fp4(w, group_size=128)     # numpy in -> numpy out
    rp, rs = ofp4.quantize_fp4(w, 128)
    assert np.array_equal(packed, rp)
    assert np.array_equal(scales.view(np.uint16), rs.view(np.uint16))


def test_pack_u4_vs_oracle(rng):
    import mmfp4
    w = rng.normal(0, 0.02, (256, 1024)).astype(np.float16)
    w[0, :128] = 0.0                                   # constant group -> floor scale
    announce("pack_u4_weights random")
    packed, s, z = mmfp4.pack_u4_weights(to_dev(w), group_size=128)
    rp, rs, rz = ofp4.pack_u4_weights(w, 128)
    assert np.array_equal(to_np(packed).view(np.uint32), rp)
    assert np.array_equal(to_np(s).view(np.uint16), rs.view(np.uint16))
    assert np.array_equal(to_np(z).view(np.uint16), rz.view(np.uint16))
    back = to_np(mmfp4.unpack_u4_weights(packed, s, z))
    assert back.shape == (256, 1024)
    assert np.array_equal(back.T.view(np.uint16), ofp4.dequant_u4(rp, rs, rz, 128).view(np.uint16))


CAL_CASES = ["cal_p999_f32", "cal_p90_small_f16", "cal_large_sf03_f32", "cal_small_sf1_g32_f32",
             "cal_p50_g8_f32", "cal_p99_crafted_f32", "cal_p37_quarter_f16", "cal_f64_blend_f32"]


@pytest.mark.parametrize("name", CAL_CASES)
def test_quantize_fp4_calibrated_matches_reference_vectors(name):
    """quantize_fp4(activation_ranges=...) on the GPU: codes and scales
    bit-identical to the reference's calibration-aware branch
    (quantize_fp4.py:205-256) and to the oracle."""
    import mmfp4
    d = np.load(GOLD)
    pct, sf, a_min, a_max = d[f"{name}__cal"]
    ar = {"percentile": float(pct), "smooth_factor": float(sf)}
    if not np.isnan(a_min):
        ar["input_range"] = (float(a_min), float(a_max))
    w, g = d[f"{name}__w"], int(d[f"{name}__g"])
    announce(f"quantize_fp4 calibrated golden {name}")
    packed, scales = mmfp4.quantize_fp4(w, group_size=g, activation_ranges=ar)
    assert np.array_equal(packed, d[f"{name}__packed"])
    assert np.array_equal(scales.view(np.uint16), d[f"{name}__scales"].view(np.uint16))


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("ar", [{"percentile": 99.5},
                                {"percentile": 12.5, "input_range": (-9.0, 3.0),
                                 "smooth_factor": 0.45},
                                {"percentile": 80.0, "input_range": (-0.37, 0.2),
                                 "smooth_factor": 0.8},
                                {"input_range": (0.0, 0.6)},
                                {"percentile": 100.0, "input_range": (-2.0, 0.5),
                                 "smooth_factor": 0.0}])
def test_quantize_fp4_calibrated_random_vs_oracle(rng, dtype, ar):
    import mmfp4
    w = rng.normal(0, 0.03, (96, 512)).astype(dtype)
    w[:, ::37] *= 30
    w[5, 128:256] = 0                                # an all-zero group: 1e-7 floor
    announce(f"quantize_fp4 calibrated random {dtype.__name__} {ar}")
    packed, scales = mmfp4.quantize_fp4(to_dev(w), group_size=128, activation_ranges=ar)
    rp, rs = ofp4.quantize_fp4_calibrated(w, 128, ar)
    assert np.array_equal(to_np(packed).view(np.uint32), rp)
    assert np.array_equal(to_np(scales).view(np.uint16), rs.view(np.uint16))


def test_quantize_fp4_calibrated_nan_group_and_bad_percentile(rng):
    import mmfp4
    w = rng.normal(0, 0.03, (8, 256)).astype(np.float32)
    w[3, 7] = np.nan
    ar = {"percentile": 90.0, "input_range": (-0.5, 0.5), "smooth_factor": 0.5}
    announce("quantize_fp4 calibrated NaN group")
    with np.errstate(invalid="ignore"):
        rp, rs = ofp4.quantize_fp4_calibrated(w, 128, ar)
    packed, scales = mmfp4.quantize_fp4(w, group_size=128, activation_ranges=ar)
    assert np.isnan(scales[0, 3]) and np.isnan(rs[0, 3])
    assert np.array_equal(np.isnan(scales), np.isnan(rs))
    ok = ~np.isnan(rs)
    assert np.array_equal(scales[ok].view(np.uint16), rs[ok].view(np.uint16))
    assert np.array_equal(packed, rp)
    with pytest.raises(ValueError):
        mmfp4.quantize_fp4(w, group_size=128, activation_ranges={"percentile": 101.0})
    # the weight-only path on the same NaN group: NaN scale, codes 8 (numpy's
    # clip keeps NaN and argmin over all-NaN distances returns index 0)
    with np.errstate(invalid="ignore"):
        rp, rs = ofp4.quantize_fp4(w, 128)
    packed, scales = mmfp4.quantize_fp4(w, group_size=128)
    assert np.array_equal(packed, rp)
    assert np.array_equal(np.isnan(scales), np.isnan(rs))
    assert np.all(ofp4.unpack_nibbles(rp)[:128, 3] == 8)


def _crafted(rng, n, k, dtype):
    """Weights with ties, signed zeros, subnormals, NaN / inf, a zero row and a
    constant row (float32 also extreme exponents)."""
    w = rng.normal(0, 0.02, (n, k)).astype(dtype)
    w[0] = 0
    w[min(1, n - 1)] = 0.25
    w.flat[5 % w.size::97] = -0.0
    w.flat[11 % w.size::101] = 6e-8
    ties = np.array([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0, 6.0], dtype)
    w[n // 2, :8] = ties
    w[n // 2, :8][::2] *= -1
    if n > 4:
        w[n - 1, k // 2], w[n - 2, 0], w[n - 2, k - 1] = np.nan, np.inf, -np.inf
        if dtype == np.float32:
            w[n - 3, ::3], w[n - 4, ::2], w[n - 4, 1::2] = 3e38, 1e-42, -1e-42
    return w


# 8 * 2^i up to 512 run the tiled quantizer; 24 and 1024 the per-group one.
@pytest.mark.parametrize("N,K,g", [(1, 8, 8), (63, 512, 16), (65, 520, 8), (64, 1536, 512),
                                   (130, 1152, 128), (66, 544, 32), (33, 768, 256),
                                   (70, 576, 64), (40, 72, 24), (9, 2048, 1024),
                                   (8200, 520, 8), (16390, 480, 32), (4106, 1664, 128)])
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_quantizers_edges(rng, N, K, g, dtype):
    """Blocks of 4 rows (small matrices) and of 64, ends inside a block or a word
    group, and the per-group kernels."""
    import mmfp4
    w = _crafted(rng, N, K, dtype)
    announce(f"quantizers N={N} K={K} g={g} {dtype.__name__}")
    with np.errstate(all="ignore"):
        rp, rs = ofp4.quantize_fp4(w, g)
    for view in (0, 1):       # view 1: rows of a tensor that is not 16-byte aligned
        t = to_dev(w)
        if view:
            t = torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(N, K)
        packed, s = mmfp4.quantize_fp4(t, group_size=g)
        assert np.array_equal(to_np(packed).view(np.uint32), rp)
        assert np.array_equal(to_np(s).view(np.uint16), rs.view(np.uint16))
    if dtype == np.float16:
        # the reference's uint32 cast of a NaN code is undefined: finite weights
        w = np.nan_to_num(w, nan=0.01, posinf=0.03, neginf=-0.02)
        rp, rs, rz = ofp4.pack_u4_weights(w, g)
        packed, s, z = mmfp4.pack_u4_weights(to_dev(w), group_size=g)
        assert np.array_equal(to_np(packed).view(np.uint32), rp)
        assert np.array_equal(to_np(s).view(np.uint16), rs.view(np.uint16))
        assert np.array_equal(to_np(z), rz)


@pytest.mark.parametrize("K,N", [(64, 1), (64, 4), (64, 64), (64, 255), (64, 1020), (544, 4096),
                                 (512, 4096), (1024, 2052), (4096, 516), (8224, 260)])
def test_dequant_widths(rng, K, N):
    """Four columns per thread (N % 4 == 0, from 65536 such threads), with whole lines
    (N % 64 == 0) and without, and one."""
    import mmfp4
    g = 32
    packed = rng.integers(0, 2**32, (K // 8, N), dtype=np.uint64).astype(np.uint32)
    s = rng.normal(0, 0.01, (K // g, N)).astype(np.float16)
    s[0, 0], s[-1, N - 1] = np.inf, np.nan
    z = rng.integers(0, 16, (K // g, N)).astype(np.float16)
    announce(f"dequant K={K} N={N}")
    out = to_np(mmfp4.dequant_fp4(to_dev(packed), to_dev(s), K, N, g))
    assert np.array_equal(out.view(np.uint16), ofp4.dequant_fp4(packed, s, g).view(np.uint16))
    out = to_np(mmfp4.dequant_int4(to_dev(packed), to_dev(s), to_dev(z), K, N, g))
    assert np.array_equal(out.view(np.uint16), ofp4.dequant_u4(packed, s, z, g).view(np.uint16))


@pytest.mark.parametrize("e", [38, 39, 40, 41, 69, 70, 71, 90, 100, 101, 126])
def test_quantize_fp4_wide_float32_groups(rng, e):
    """float32 groups whose largest weight is 2^e beside small ones of both signs,
    down to and past 2^-80: around the divisor limit of the tiled quantizer, and
    where the quotient underflows to -0 (code 0)."""
    import mmfp4
    N, K, g = 64, 1024, 128
    w = np.ldexp(rng.uniform(1, 2, (N, K)), rng.integers(-82, min(e, 40), (N, K))).astype(np.float32)
    w[:, ::3] = np.ldexp(1.0, -80)
    w[:, 1::16] = np.ldexp(1.0, -60)
    w *= rng.choice([-1, 1], (N, K)).astype(np.float32)
    w[:, ::g] = np.ldexp(1.0, e)
    announce(f"quantize float32 absmax 2^{e}")
    with np.errstate(all="ignore"):
        rp, rs = ofp4.quantize_fp4(w, g)
    packed, s = mmfp4.quantize_fp4(to_dev(w), group_size=g)
    assert np.array_equal(to_np(s).view(np.uint16), rs.view(np.uint16))
    assert np.array_equal(to_np(packed).view(np.uint32), rp)


def _queued_us(call, n=40):
    """Median GPU time of a call with the launches queued ahead."""
    call()
    times = []
    for _ in range(7):
        torch.cuda._sleep(1_000_000)
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(n):
            call()
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b) * 1000 / n)
    return sorted(times)[3]


@pytest.mark.parametrize("N,K,g", [(33, 1024, 8), (4, 512, 8), (256, 256, 32)])
def test_small_quantizers_tiled_form_is_not_slower(N, K, g):
    """Small matrices through the tiled quantizers and (weights that are not 16-byte
    aligned) the per-group ones: INT4 33 x 1024 in groups of 8 2.4 against 2.6 us; 9.0
    in blocks of 64 rows."""
    import mmfp4
    lib = mmfp4._lib
    w = (torch.randn(N * K + 8, device="cuda") * 0.02).half()
    p = torch.empty(K // 8, N, device="cuda", dtype=torch.int32)
    s, z = (torch.empty(K // g, N, device="cuda", dtype=torch.float16) for _ in range(2))
    st = lib.stream_of(s)

    def u4(first):
        lib.call("mm_u4_quantize", lib.ptr(w[first:]), N, K, g, lib.ptr(p), lib.ptr(s),
                 lib.ptr(z), st)

    def fp4(first):
        lib.call("mm_fp4_quantize", lib.ptr(w[first:]), 0, N, K, g, lib.ptr(p), lib.ptr(s), st)

    announce(f"small quantizers N={N} K={K} g={g}")
    for quantize in (u4, fp4):
        tiled, per_group = (_queued_us(lambda f=f: quantize(f)) for f in (0, 1))
        assert tiled < 1.2 * per_group, f"{quantize.__name__}: {tiled:.2f}, {per_group:.2f} us"


@pytest.mark.parametrize("K,N", [(5376, 4516), (1024, 100)])
def test_dequant_wide_form_is_not_slower(K, N):
    """Operands that allow four words per thread against one word per thread (scales
    that are not 8-byte aligned) into a destination that is used again.  At a width
    whose rows end inside a cache line 13.0 against 14.1 us, 16.4 with stores that
    bypassed the caches; a small matrix takes one word per thread either way, 2.0 us
    (2.4 with four)."""
    import mmfp4
    g = 32
    p = torch.randint(-2**31, 2**31 - 1, (K // 8, N), device="cuda", dtype=torch.int32)
    s = torch.full((K // g * N + 4,), 0.01, device="cuda", dtype=torch.float16)
    z = torch.full((K // g, N), 7.0, device="cuda", dtype=torch.float16)
    out = torch.empty((K, N), device="cuda", dtype=torch.float16)
    lib = mmfp4._lib

    def us(first):
        sv, st = s[first:first + K // g * N], lib.stream_of(out)
        return _queued_us(lambda: lib.call("mm_u4_dequant", lib.ptr(p), lib.ptr(sv), lib.ptr(z),
                                           lib.ptr(out), K, N, g, st))

    announce(f"dequant forms K={K} N={N}")
    one, four = us(1), us(0)
    assert four < 1.12 * one, f"{four:.2f} us with four words per thread, {one:.2f} with one"
