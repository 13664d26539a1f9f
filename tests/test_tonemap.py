"""sRGB tonemap (src/kernel/tonemap.cu:7-39): the oracle's restatement against the closed-form
sRGB transfer function of IEC 61966-2-1 evaluated in double, the special values, the PNG
round trip; on the GPU, cx_tonemap against the oracle bit for bit."""
import os

import numpy as np
import pytest

from crisoptix_amd import image


def srgb_closed_form(c):
    c = np.asarray(c, np.float64)
    with np.errstate(invalid="ignore"):
        return np.where(c < 0.0031308, 12.92 * c, 1.055 * np.power(np.maximum(c, 0.0), 1.0 / 2.4) - 0.055)


def test_oracle_tonemap_matches_srgb_curve(orc):
    rng = np.random.default_rng(0)
    c = np.concatenate([np.linspace(0.0, 1.2, 200001), rng.random(100000) * 2.0,
                        [0.0031308, np.nextafter(np.float32(0.0031308), 0), 1.0, 1e-8]]).astype(np.float32)
    got = orc.tonemap(c).astype(np.int64)
    v = np.clip(srgb_closed_form(c), 0.0, 1.0) * 255.0
    exp = np.floor(v).astype(np.int64)
    # away from the truncation boundaries the float pipeline must give the exact byte
    safe = np.abs(v - np.round(v)) > 1e-4
    assert np.array_equal(got[safe], exp[safe])
    assert np.max(np.abs(got - exp)) <= 1
    # the curve is continuous at the breakpoint and monotone
    assert np.all(np.diff(orc.tonemap(np.sort(c)).astype(np.int64)) >= 0)


def test_oracle_tonemap_special_values(orc):
    c = np.asarray([-1.0, -0.0, 0.0, np.inf, -np.inf, np.nan, 1.0, 100.0], np.float32)
    got = orc.tonemap(c)
    # negative: 12.92 c < 0 clamps to 0; +inf: the lerp of 12.92 inf * 0 is NaN -> 0; NaN -> 0;
    # 1.0: 1.055f - 0.055f rounds to 1 - 2^-24 in float, so 255 x that truncates to 254 (the
    # reference's arithmetic; only values a little above 1 reach 255)
    assert list(got) == [0, 0, 0, 0, 0, 0, 254, 255]


def test_png_round_trip(tmp_path):
    rng = np.random.default_rng(1)
    a = rng.integers(0, 256, (7, 13, 3), dtype=np.uint8)
    p = str(tmp_path / "x.png")
    image.write_png(p, a)
    assert np.array_equal(image.read_png(p), a)
    with open(p, "rb") as f:
        assert f.read(8) == b"\x89PNG\r\n\x1a\n"


@pytest.mark.gpu
def test_gpu_tonemap_bit_exact(orc, cx_runtime, cx_ctx):
    rng = np.random.default_rng(2)
    c = np.concatenate([rng.random(300000) * 1.5, rng.standard_normal(1000) * 10, np.linspace(0, 0.01, 10000),
                        [np.inf, -np.inf, np.nan, 0.0031308]]).astype(np.float32)
    d = cx_runtime.DeviceArray.from_numpy(c)
    got = cx_runtime.tonemap(cx_ctx, d)
    assert np.array_equal(got, orc.tonemap(c))


@pytest.mark.gpu
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 1023, 1024, 1025, 300_001])
def test_gpu_tonemap_sizes_and_alignment(n, shift, orc, cx_runtime, cx_ctx):
    """Output words cut at either end (the bytes beyond them stay as they are), input and output at
    any alignment that their types allow, values on both sides of every step of the bytes."""
    from crisoptix_amd.runtime import DeviceArray, lib, synchronize
    steps = (((np.arange(1, 256) / 255.0 + 0.055) / 1.055) ** 2.4).astype(np.float32)
    ulps = steps.view(np.int32)[:, None] + np.arange(-40, 41, dtype=np.int32)
    special = np.array([0.0, -0.0, -1.0, np.nan, np.inf, -np.inf, 1.0, 1.001, 0.0031308, 3e37, 1e-45, 3.4e38, 12.0],
                       np.float32)
    c = np.resize(np.concatenate([special, ulps.view(np.float32).ravel(),
                                  np.random.default_rng(5).random(9000, np.float32) * 1.1]), n)
    hdr = DeviceArray.from_numpy(np.concatenate([np.zeros(shift, np.float32), c]))
    ldr = DeviceArray.from_numpy(np.full(n + 16, 0xA5, np.uint8))
    cx_ctx.check(lib().cx_tonemap(cx_ctx.h, hdr.ptr + 4 * shift, ldr.ptr + 4 + shift, n, None), "cx_tonemap")
    synchronize()
    got = ldr.numpy()
    assert np.array_equal(got[4 + shift:4 + shift + n], orc.tonemap(c))
    assert np.all(got[:4 + shift] == 0xA5) and np.all(got[4 + shift + n:] == 0xA5)


@pytest.mark.gpu
def test_gpu_tonemap_every_float_of_the_curve(orc, cx_runtime, cx_ctx):
    """Every float that takes the power (0.0031308 to 1.001, beyond which the clamp gives 255), where
    the kernel estimates the byte and falls back on the double power beside its steps, and every 97th
    of all floats, NaN payloads and both infinities among them."""
    from concurrent.futures import ThreadPoolExecutor
    first, last = (int(np.float32(x).view(np.uint32)) for x in (0.0031308, 1.001))
    curve = np.arange(first - 64, last + 64, dtype=np.uint32)
    parts = np.array_split(curve, 8) + np.array_split(np.arange(0, 2**32, 97, dtype=np.uint64).astype(np.uint32), 8)
    with ThreadPoolExecutor(8) as ex:
        for i, (part, ref) in enumerate(zip(parts, ex.map(lambda p: orc.tonemap(p.view(np.float32)), parts))):
            got = cx_runtime.tonemap(cx_ctx, cx_runtime.DeviceArray.from_numpy(part.view(np.float32)))
            bad = np.flatnonzero(got != ref)
            print(f"part {i}: {part.size} floats, {bad.size} differ", flush=True)
            assert bad.size == 0, part[bad[:8]]


@pytest.mark.gpu
def test_gpu_tonemap_of_a_white_image_takes_little_longer(orc, cx_runtime, cx_ctx):
    """A clamped image is 1.0 over whole regions, a value next to a step of the byte whose power is known:
    it takes little longer than a grey one (5 times as long where every value took the double power)."""
    import time
    times = {}
    for v in (0.5, 1.0):
        d = cx_runtime.DeviceArray.from_numpy(np.full(8_000_000, v, np.float32))
        out = cx_runtime.DeviceArray((8_000_000,), np.uint8)
        t = []
        for _ in range(8):
            cx_runtime.synchronize()
            t0 = time.perf_counter()
            for _ in range(20):
                cx_ctx.check(cx_runtime.lib().cx_tonemap(cx_ctx.h, d.ptr, out.ptr, 8_000_000, None), "cx_tonemap")
            cx_runtime.synchronize()
            t.append(time.perf_counter() - t0)
        times[v] = min(t)
        assert np.all(out.numpy() == orc.tonemap(np.float32([v]))[0])
    print({k: f"{x / 20 * 1e6:.1f} us" for k, x in times.items()})
    assert times[1.0] < 3.0 * times[0.5], times
