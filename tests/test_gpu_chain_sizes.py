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


@pytest.mark.parametrize("h,w", PLANS)
@pytest.mark.parametrize("variant", [_lib.PCE_REFERENCE, _lib.PCE_TEXTBOOK])
def test_pce_plans(variant, h, w, rng):
    """Relative PCE error <= 1e-4, the bound of every other size."""
    if h * w <= 121 or min(h, w) < 11:
        pytest.skip("the window covers the plane or wraps onto itself")
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
