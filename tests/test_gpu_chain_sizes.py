"""The extraction chain at sizes where its kernels change form: odd and even
widths (column means alone, or with row means, in the zero-mean), widths off
the multiple of 4 of the row-walking FastNoise, heights around its band
lengths, and images on both sides of the sizes that choose the band.

Tolerance: 2e-5 of the largest magnitude of the expected pattern (two 2-D
FP32 FFTs), as for every other size of the chain.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import prnu_oracle as O  # noqa: E402
from rocket_amd import _lib, csi  # noqa: E402

pytestmark = pytest.mark.gpu


def chain(img, fmt, spectrum=False):
    h, w = img.shape[:2]
    f = csi.PRNUFilter(h, w, apply_spectral_filter=spectrum)
    out = torch.empty(f.get_output_size() // 4, device="cuda")
    f.apply_gpu(torch.from_numpy(img).cuda(), out, fmt)
    got = out.cpu().numpy().astype(np.float64)
    f.cleanup()
    return got


@pytest.mark.parametrize("h,w", [(3, 8), (9, 8), (8, 250), (27, 75), (16, 45), (50, 54), (25, 256), (75, 500),
                                 (1080, 640), (1620, 1600)])
@pytest.mark.parametrize("fmt", ["rgb8", "gray8", "float32"])
def test_chain_forms(h, w, fmt, rng):
    if fmt != "rgb8" and h * w > 1 << 19:
        pytest.skip("one format is enough at the large sizes")
    gray = rng.integers(0, 256, size=(h, w), dtype=np.uint8)
    if fmt == "rgb8":
        img = rng.integers(0, 256, size=(h, w, 3), dtype=np.uint8)
        want, code = O.prnu_pattern(img), _lib.INPUT_RGB8
    elif fmt == "gray8":
        img, want, code = gray, O.prnu_pattern(gray), _lib.INPUT_GRAY8
    else:
        img, code = gray.astype(np.float32), _lib.INPUT_FLOAT32
        want = O.wiener(O.zeromean(O.fastnoise(img)))
    got = chain(img, code).reshape(h, w)
    assert np.abs(got - want).max() <= 2e-5 * max(np.abs(want).max(), 1e-30)


def striped(h, w, kind, patch, seed):
    """A frame whose rows are constant, with one textured patch."""
    r = np.random.default_rng(seed)
    y = np.arange(h)
    row = {"sine": 128 + 100 * np.sin(2 * np.pi * y / 37.3), "bars": np.where(y // 2 % 2, 230, 20),
           "noise": r.integers(0, 256, h)}[kind]
    img = np.repeat(np.round(row)[:, None], w, axis=1).astype(np.uint8)
    img[h // 3:h // 3 + patch, w // 4:w // 4 + patch] = r.integers(0, 256, (patch, patch))
    return img


@pytest.mark.parametrize("h,w,kind,patch", [(1500, 2000, "bars", 8), (1500, 2000, "noise", 8), (1500, 2000, "sine", 64),
                                            (1000, 1500, "bars", 8), (1080, 1920, "bars", 8), (240, 1000, "bars", 8),
                                            (240, 1800, "noise", 8), (1536, 2048, "noise", 8), (1536, 2048, "bars", 64),
                                            (1024, 1024, "noise", 16), (75, 500, "noise", 4)])
def test_striped_frames(h, w, kind, patch):
    """Frames whose row means carry nearly all of the energy before the
    zero-mean, which the Wiener variance must not see."""
    img = striped(h, w, kind, patch, h + w)
    want = O.prnu_pattern(img)
    got = chain(img, _lib.INPUT_GRAY8).reshape(h, w)
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


@pytest.mark.parametrize("h,w", [(240, 1000), (1000, 1500), (96, 60)])
def test_stripes_alone(h, w):
    """Row-constant frames: the exact pattern is zero and what is left is the
    rounding of a transform of values up to 1, 2^-24 per value and level (13
    levels at most), times a scale of at most 1.  (Zero exactly, the scale is
    0 / 0: NaN.)"""
    for seed in range(6):
        for kind in ("noise", "sine", "bars"):
            img = striped(h, w, kind, 0, seed)
            got = chain(img, _lib.INPUT_GRAY8)
            assert np.isnan(got).all() or np.abs(got).max() <= 4 * 13 * 2.0 ** -24


def test_wiener_infinite_power_beside_a_box():
    """Two waves, the first of a power past FP32.  The box of the second holds
    the first's bin on one side (variance infinite, scale 0) and on the mirrored
    side, cut by the spectrum's edge, does not (variance P / 81): the first
    vanishes, the second keeps half of that side's scale.  Tolerance 1e-3 of
    what is left: the transforms' rounding, 2^-24 of the first wave per bin,
    is some 1e-4 of it."""
    h, w, n = 48, 64, 48 * 64
    y, x = np.mgrid[0:h, 0:w]
    a, b = 1.3e16, 1.0e16
    wave = np.cos(2 * np.pi * (21 * x / w + y / h))
    img = (a * np.cos(2 * np.pi * 20 * x / w) + b * wave).astype(np.float32)
    assert (n * a / 2) ** 2 > float(np.finfo(np.float32).max) > (n * b / 2) ** 2
    var = np.sum(img.astype(np.float64) ** 2) * n / (n - 1)
    want = 0.5 * var / ((n * b / 2) ** 2 / 81) * b * wave
    f = csi.PRNUFilter(h, w)
    t = torch.from_numpy(img.ravel()).cuda()
    f.get_wiener_filter().apply_gpu(t)
    f.cleanup()
    assert np.abs(t.cpu().numpy().reshape(h, w) - want).max() <= 1e-3 * np.abs(want).max()


# heights and widths of every plan of the column strips (64 threads per column
# below 1024 rows, 128 up to 2048, 256 up to 4096, 512 above) and of the rows,
# with an odd number of columns, fewer columns than a strip, and one radix alone
PLANS = [(16, 20), (15, 9), (600, 45), (960, 10), (1200, 18), (2000, 27), (2048, 6), (2250, 8), (4096, 4), (4374, 6),
         (8100, 4), (1536, 15), (1024, 30), (20, 1800), (9, 2048), (12, 2500), (6, 7500), (10, 1536)]


@pytest.mark.parametrize("h,w", PLANS)
def test_wiener_and_spectrum_plans(h, w, rng):
    x = O.zeromean(rng.normal(size=(h, w))).astype(np.float32)
    f = csi.PRNUFilter(h, w, apply_spectral_filter=True)
    t = torch.from_numpy(x.ravel()).cuda()
    spec = torch.empty(2 * h * (w // 2 + 1), device="cuda")
    f.get_spectral_filter().apply_gpu(t, spec)
    want = O.spectrum(x)
    got = spec.cpu().numpy().view(np.complex64).reshape(h, w // 2 + 1)
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()
    f.get_wiener_filter().apply_gpu(t)
    want = O.wiener(x)
    assert np.abs(t.cpu().numpy().reshape(h, w) - want).max() <= 2e-5 * np.abs(want).max()
    f.cleanup()


@pytest.mark.parametrize("h,w", [(24, 512), (25, 500), (500, 540)])
def test_batch_equals_single_across_the_stencil(h, w, rng):
    """24 frames fill the chip with the variance stencil's long tiles, one frame
    takes the short ones: the same bits."""
    count = max(24, -(-512 // (-(-h // 64) * ((w // 2 + 128) // 128))))
    imgs = torch.from_numpy(rng.integers(0, 256, size=(count, h * w), dtype=np.uint8)).cuda()
    f = csi.PRNUFilter(h, w)
    out, one = torch.empty((count, h * w), device="cuda"), torch.empty(h * w, device="cuda")
    f.apply_gpu_batch(imgs, out, _lib.INPUT_GRAY8)
    for i in (0, count // 2, count - 1):
        f.apply_gpu(imgs[i], one, _lib.INPUT_GRAY8)
        assert torch.equal(out[i], one)
    f.cleanup()


# PCE's forms: rows of 1024 and 2048 values in mirror pairs, shorter ones too,
# longer ones and 1536 one by one; columns of 1024 and 1536 by strips (16-byte
# and, for odd widths, 8-byte staging, a last strip of few columns), the others
# through a transpose in three size classes; even and odd numbers of rows
PCE_PLANS = [(16, 20), (600, 45), (1200, 18), (2000, 27), (1536, 15), (1024, 30), (20, 1800), (12, 2500), (12, 2048),
             (15, 2048), (15, 1024), (96, 1024), (1536, 64), (1536, 2048), (1024, 45), (16, 1536), (12, 7500),
             (2048, 24), (2250, 18), (4374, 12), (7500, 12), (8100, 12), (2048, 1536)]


@pytest.mark.parametrize("h,w", PCE_PLANS)
@pytest.mark.parametrize("variant", [_lib.PCE_REFERENCE, _lib.PCE_TEXTBOOK])
def test_pce_plans(variant, h, w, rng):
    """Relative PCE error <= 1e-4, the bound of every other size."""
    k = rng.normal(size=(h, w))
    pats = [(0.5 * k + rng.normal(size=(h, w))).astype(np.float32) for _ in range(3)]
    spec = [np.ascontiguousarray(O.spectrum(p).astype(np.complex64)) for p in pats]
    cmp = csi.PeakToCorrelationEnergy(h, w, variant)
    got = cmp.pairs([torch.from_numpy(s.view(np.float32)).cuda() for s in spec], [(0, 1), (0, 2), (1, 2)]).cpu().numpy()
    full = O.pce_reference_from_corr if variant == _lib.PCE_REFERENCE else O.pce_textbook_from_corr
    for (i, j), v in zip([(0, 1), (0, 2), (1, 2)], got):
        a, b = spec[i].astype(np.complex128), spec[j].astype(np.complex128)
        if variant == _lib.PCE_REFERENCE:
            c = np.fft.ifft2(O.cross_spectrum_reference(a, b, w)).real * (h * w)
        else:
            c = np.fft.irfft2(np.conj(a) * b, s=(h, w))
        want = full(c)[0]
        if abs(c.flat[-1]) < 0.05 * np.abs(c).std() and variant == _lib.PCE_REFERENCE:
            continue  # the scored element is nearly zero: its relative error is not bounded
        assert abs(v - want) <= 1e-4 * abs(want)
    cmp.cleanup()
