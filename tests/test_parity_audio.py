"""Parity of the output stage's kernels (kk_fir, kk_pcm16, kk_fir_pcm16)
with the oracle, through the C ABI (runtime/audio.gd:59-106,
kernels/fir.glsl:35-47, kernels/pcm16.glsl:28-46).

Bars: the FIR within fp32 summation rounding of the oracle -- both add the
taps in order, the device with a fused multiply-add per tap, the oracle with
a product and a sum rounded separately, so they differ by at most a few
units of 2^-24 * sum_k |h_k x_k| per output (held here to 4e-6 of that sum);
PCM16 of the same floats bit-exact (ties excepted: GLSL leaves them to the
implementation, the device rounds them away from zero, as the oracle
does); the fused kernel bit-exact with the two kernels in turn."""
import numpy as np
import pytest

from conftest import rng

pytestmark = pytest.mark.gpu


def fir_bound(x, h, c):
    """sum_k |h_k x_k| per output, edges clamped, in float64."""
    n, t = x.size, h.size
    xp = np.abs(x.astype(np.float64))[np.clip(np.arange(-c, n - c + t - 1), 0, n - 1)]
    return np.correlate(xp, np.abs(h.astype(np.float64)), mode="valid")


@pytest.mark.parametrize("n,t,c", [
    (2154000, 1023, -1),   # the 128-id waveform's length, the notch filter
    (167400, 1023, -1),    # the 8-id waveform
    (1000, 1023, -1),      # shorter than the filter: clamped edges on both sides
    (1, 1023, -1), (9, 7, 0), (2049, 13, 12), (4100, 8, 3), (333, 1, 0), (12345, 4096, 2047),
])
def test_fir(gpu, oracle, n, t, c):
    r = rng(40)
    x = r.normal(0, 0.3, n).astype(np.float32)
    h = oracle.notch_taps() if t == 1023 else r.normal(0, 0.1, t).astype(np.float32)
    got = gpu.to_host(gpu.ops.fir(gpu.to_device(x.reshape(1, -1)), gpu.to_device(h), c)).reshape(-1)
    cc = (t - 1) // 2 if c < 0 else c
    want = oracle.fir(x, h, cc)
    err = np.abs(got.astype(np.float64) - want)
    bound = 4e-6 * fir_bound(x, h, cc) + 1e-30
    assert (err <= bound).all(), f"max err/bound {float((err / bound).max()):.3g}"


@pytest.mark.parametrize("n,t,c", [
    (1, 32, -1), (1023, 33, 0), (1024, 49, 48), (1027, 271, 5), (5000, 1536, 1535), (5000, 4096, 3),
    (3 * 1024 + 2, 993, 0), (255, 31, 7), (256 * 4096, 300, 11), (256 * 4096 - 4097, 1023, 1022),
    (1500001, 64, 0), (2029200, 36, 35)])
def test_fir_matrix_core_tiles(gpu, oracle, n, t, c):
    """The matrix-core FIR at the edges of its tiles, of its sum's steps and
    of its range of taps, the bar as above; and an infinity or NaN reaches
    the outputs that read it, no other."""
    r = rng(43)
    x = r.normal(0, 0.3, n).astype(np.float32)
    h = r.normal(0, 0.1, t).astype(np.float32)
    cc = (t - 1) // 2 if c < 0 else c
    for special in (None, np.inf, np.nan):
        if special is not None:
            if n > 10000 or t < 32:  # (the other kernel pads its last taps)
                break
            x[n // 2] = special
        got = gpu.ops.fir(gpu.to_device(x), gpu.to_device(h), c).numpy()
        with np.errstate(all="ignore"):
            want = oracle.fir(x, h, cc)
            bound = 4e-6 * fir_bound(np.where(np.isfinite(x), x, 0), h, cc) + 1e-30
        fin = np.isfinite(want)
        np.testing.assert_array_equal(np.isnan(got[~fin]), np.isnan(want[~fin]))
        np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
        err = np.abs(got[fin].astype(np.float64) - want[fin])
        assert (err <= bound[fin]).all(), f"{special}: max err/bound {float((err / bound[fin]).max()):.3g}"


def fma_chain(h, x):
    """sum_k h[k] x[k:k + m] in order, one correctly rounded fused
    multiply-add a term: the product is exact in float64, and its sum with
    the accumulator is rounded to odd there, so that the rounding to float32
    is that of the exact sum."""
    m = x.size - h.size + 1
    acc = np.zeros(m, np.float32)
    for k in range(h.size):
        p = np.float64(h[k]) * x[k:k + m].astype(np.float64)
        a = acc.astype(np.float64)
        s = p + a
        b = s - p
        err = (p - (s - b)) + (a - b)  # p + a - s, exactly
        even = (s.view(np.int64) & 1) == 0
        s = np.where((err != 0) & even, np.nextafter(s, np.where(err > 0, np.inf, -np.inf)), s)
        acc = s.astype(np.float32)
    return acc


@pytest.mark.parametrize("n,t,c", [
    (3000, 31, 4), (3000, 32, -1), (3001, 49, 7), (3003, 271, -1), (2999, 1023, -1), (2500, 4096, 100),
    (1500001, 1023, -1),   # two tiles a wave
    (2029203, 1023, -1), (1060001, 4096, -1), (3200003, 40, 3), (4000001, 255, 17)])  # four, and other costs
def test_fir_is_the_tap_chain(gpu, n, t, c):
    """The FIR, fp32 and PCM16, bit for bit the chain of fused multiply-adds
    in tap order, at the waveform's edges and inside it."""
    r = rng(55)
    x = r.normal(0, 0.3, n).astype(np.float32)
    h = r.normal(0, 0.05, t).astype(np.float32)
    dx, dh = gpu.to_device(x), gpu.to_device(h)
    got = gpu.ops.fir(dx, dh, c).numpy()
    cc = (t - 1) // 2 if c < 0 else c
    for lo in sorted({0, n // 2, max(0, n - 2500)}):
        hi = min(n, lo + 2500)
        piece = x[np.clip(np.arange(lo - cc, hi - cc + t - 1), 0, n - 1)]
        np.testing.assert_array_equal(got[lo:hi].view(np.uint32), fma_chain(h, piece).view(np.uint32))
    fused = gpu.to_host(gpu.ops.fir_pcm16(dx, dh, c, 0.9))
    np.testing.assert_array_equal(fused, gpu.to_host(gpu.ops.pcm16(gpu.ops.fir(dx, dh, c), 0.9)))


def test_fir_notch_removes_the_hop_tones(gpu, oracle):
    """A waveform carrying the iSTFT's 4800 / 9600 Hz ring: the device filter
    takes both tones down by at least 40 dB and leaves a 1 kHz tone within
    0.1 dB (away from the edges)."""
    t = np.arange(48000) / 24000.0
    ring = (0.1 * np.sin(2 * np.pi * 4800 * t) + 0.05 * np.sin(2 * np.pi * 9600 * t)).astype(np.float32)
    voice = (0.3 * np.sin(2 * np.pi * 1000 * t)).astype(np.float32)
    h = gpu.to_device(oracle.notch_taps())
    y_ring = gpu.to_host(gpu.ops.fir(gpu.to_device(ring), h))[2000:-2000]
    y_voice = gpu.to_host(gpu.ops.fir(gpu.to_device(voice), h))[2000:-2000]
    rms = lambda v: float(np.sqrt(np.mean(np.asarray(v, np.float64) ** 2)))
    assert 20 * np.log10(rms(y_ring) / rms(ring[2000:-2000])) < -40.0
    assert abs(20 * np.log10(rms(y_voice) / rms(voice[2000:-2000]))) < 0.1


@pytest.mark.parametrize("n", [2154000, 167400, 9, 8, 1, 7])
def test_pcm16(gpu, oracle, n):
    r = rng(41)
    x = r.normal(0, 0.6, n).astype(np.float32)  # ~10% beyond +-1: the clamp
    x[: min(n, 4)] = np.array([1.0, -1.0, 2.5, -7.0], np.float32)[: min(n, 4)]
    for gain in (1.0, 0.7):
        raw = gpu.to_host(gpu.ops.pcm16(gpu.to_device(x), gain))
        assert raw.dtype == np.uint8 and raw.size == 2 * n
        np.testing.assert_array_equal(raw.view("<i2"), oracle.pcm16(x, gain))


def test_pcm16_ties_round_away_from_zero(gpu, oracle):
    """Values whose scaled sample is an exact .5: the device (and the oracle)
    round away from zero; GLSL's round() may go either way there, so these
    are parity unpinned against the reference."""
    k = np.array([0, 1, 2, 100, 16383], np.float64)
    x = np.concatenate([(k + 0.5) / 32767.0, -(k + 0.5) / 32767.0]).astype(np.float32)
    s = x.astype(np.float64) * 32767.0
    ties = s == np.floor(s) + 0.5
    got = gpu.to_host(gpu.ops.pcm16(gpu.to_device(x))).view("<i2")
    np.testing.assert_array_equal(got, oracle.pcm16(x))
    assert ties.any()
    np.testing.assert_array_equal(got[ties], (np.sign(s) * np.ceil(np.abs(s)))[ties].astype(np.int16))


@pytest.mark.parametrize("n", [2154000, 1000, 3])
def test_fir_pcm16_fused(gpu, oracle, n):
    r = rng(42)
    x = gpu.to_device(r.normal(0, 0.8, n).astype(np.float32))
    h = gpu.to_device(oracle.notch_taps())
    fused = gpu.to_host(gpu.ops.fir_pcm16(x, h, -1, 0.9))
    two = gpu.to_host(gpu.ops.pcm16(gpu.ops.fir(x, h), 0.9))
    np.testing.assert_array_equal(fused, two)


def test_output_stage_errors(gpu, oracle):
    kk = gpu
    x = kk.to_device(np.zeros(100, np.float32))
    with pytest.raises(kk._lib.KKError, match="taps"):
        kk.ops.fir(x, kk.to_device(np.zeros(4097, np.float32)))
    with pytest.raises(kk._lib.KKError, match="center"):
        kk.ops.fir(x, kk.to_device(np.zeros(5, np.float32)), 5)
    with pytest.raises(kk._lib.KKError, match="fp32"):
        kk.ops.pcm16(kk.to_device(np.zeros(10, np.int32)))
