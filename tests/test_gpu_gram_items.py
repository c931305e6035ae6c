"""The Gram kernels at the counts and lengths where their work items change
form: one 128-pattern quarter (four slabs at once), three quarters (two), five
(one), nine (four, in the second of two one-quarter items), a single short
slab, ragged last slabs and K blocks.

Tolerances against FP64: 1e-5 for FP32 and split-BF16 products; FP16 and FP8
values are rounded once per element (relative 2^-11 and 2^-4, rms 0.29 and
0.036 / 2^-4 of that), so an entry errs by that share of 1/sqrt(n) for
unrelated patterns and of the entry for related ones: 6 sigma of sqrt(2) such
roundings, with the diagonal's bias 2 * rms^2.
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import prnu_oracle as O  # noqa: E402
from rocket_amd import _lib, csi  # noqa: E402
from test_gpu_ncc import patterns  # noqa: E402

pytestmark = pytest.mark.gpu


def tolerance(fmt, n):
    rms = {"fp16": 2.0 ** -11, "fp8": 0.04}.get(fmt)
    return 1e-5 if rms is None else 6 * rms * np.sqrt(2.0 / n) * 2 + 2 * rms * rms + 1e-5


@pytest.mark.parametrize("fmt", ["split_bf16", "fp32", "fp16", "fp8"])
@pytest.mark.parametrize("count,h,w", [(1, 8, 9), (5, 20, 21), (120, 164, 167), (128, 100, 100), (300, 161, 150),
                                       (384, 33, 64), (600, 40, 41), (1100, 30, 31)])
def test_items(fmt, count, h, w):
    p = patterns(count, h, w, 4, seed=900 + count, gain=0.3)
    want = O.ncc_matrix(p.cpu().numpy())
    tol = tolerance(fmt, h * w)
    gram = csi.GramNCC(h, w)
    store = csi.PatternStore(h * w, count + 2, fmt)
    store.put(p, first_slot=2)
    for slabs in (0, 1, 3, 7, 300):
        cfg = (ctypes.c_int32 * 3)(slabs, 1, 0)
        _lib.call("prnu_gram_set_config", gram._ctx.handle, _lib.PRECISIONS[fmt], cfg)
        got = store.gram(gram, count, 2).cpu().numpy()
        assert np.abs(got - want).max() <= tol
        assert np.array_equal(got, got.T)
        if fmt != "fp16":
            assert np.abs(gram.ncc(p, fmt).cpu().numpy() - want).max() <= tol
    store.close()
    gram.close()


@pytest.mark.parametrize("slab_blocks", [1, 4, 9, 40])
def test_split_item_keeps_the_slabs(slab_blocks):
    """The same slabs give the same bits whether a pair lies in a set of one
    quarter (four slabs at once, where there are more slabs than CUs) or of two
    (one at a time)."""
    h, w, n = 240, 440, 240 * 440
    p = patterns(200, h, w, 4, seed=77, gain=0.3)
    gram = csi.GramNCC(h, w)
    store = csi.PatternStore(n, 200, "split_bf16")
    store.put(p)
    plans = [csi.GramPlan(gram, [(store, 0, c)], slab_values=32 * slab_blocks) for c in (100, 200)]
    small, large = (pl.run()[0].cpu().numpy() for pl in plans)
    assert np.array_equal(small, large[:100, :100])
    plans[0].persistent = True
    assert np.array_equal(plans[0].run()[0].cpu().numpy(), small)
    for pl in plans:
        pl.close()
    store.close()
    gram.close()


@pytest.mark.parametrize("fmt", ["split_bf16", "fp32", "fp16", "fp8"])
@pytest.mark.parametrize("count", [120, 300])
@pytest.mark.parametrize("blocks,per_slab", [(2001, 7), (1201, 4), (900, 3)])
def test_split_items(fmt, count, blocks, per_slab):
    """Split items of several stages with short last slabs and groups: near
    FP64, and the same bits by every way of loading, as a plan's set and from a
    persistent launch."""
    values = {"split_bf16": 32, "fp32": 32, "fp16": 64, "fp8": 128}[fmt]
    n = (values * blocks - 5) // 3 * 3
    p = patterns(count, n // 3, 3, 4, seed=blocks + count, gain=0.3)
    want = O.ncc_matrix(p.cpu().numpy())
    gram = csi.GramNCC(n // 3, 3)
    store = csi.PatternStore(n, count + 2, fmt)
    store.put(p, first_slot=2)
    slabs = -(-blocks // per_slab)
    assert slabs > 256  # more items than CUs: the last one takes several slabs
    got = []
    for variant in (0, 1, 2):
        cfg = (ctypes.c_int32 * 3)(slabs, 1, variant)
        _lib.call("prnu_gram_set_config", gram._ctx.handle, _lib.PRECISIONS[fmt], cfg)
        got.append(store.gram(gram, count, 2).cpu().numpy())
    plan = csi.GramPlan(gram, [(store, 2, count)], slab_values=values * per_slab)
    for persistent in (False, True):
        plan.persistent = persistent
        got.append(plan.run()[0].cpu().numpy())
    plan.close()
    store.close()
    gram.close()
    assert np.abs(got[0] - want).max() <= tolerance(fmt, n)
    for g in got[1:]:
        assert np.array_equal(g, got[0])


@pytest.mark.parametrize("fmt", ["split_bf16", "fp32", "fp16", "fp8"])
@pytest.mark.parametrize("count,n,first,offset", [(1, 6, 0, 0), (9, 1023, 2, 0), (8, 1024, 0, 0), (17, 1029, 3, 1),
                                                  (5, 5000, 1, 3), (4, 8193, 0, 1), (6, 20000, 2, 0)])
def test_put_edges(fmt, count, n, first, offset):
    """Inserts around the packing's 8 patterns and 1024 values, with pattern
    rows off 16-byte alignment: the stored statistics (FP64 sums of FP32
    products: 1e-10), slots around the range untouched, and the same blocks and
    statistics as one pattern put at a time (bytes equal; up to four patterns a
    call take eight pieces of one pattern to a workgroup)."""
    g = torch.Generator(device="cuda").manual_seed(n + count)
    rows = [torch.randn(n + offset, generator=g, device="cuda")[offset:] for _ in range(count)]
    stores = [csi.PatternStore(n, first + count + 2, fmt) for _ in range(2)]
    stores[0].put(rows, first_slot=first)
    for i, r in enumerate(rows):
        stores[1].put([r], first_slot=first + i)
    images = []
    for s in stores:
        img = torch.empty(s.image_bytes(first + count + 2), dtype=torch.uint8)
        s.save(0, first + count + 2, img)
        images.append(img.numpy())
    blocks = len(images[0]) - (first + count + 2) * 24   # the slots past and before `first` hold no statistics yet
    assert np.array_equal(images[0][:blocks], images[1][:blocks])
    assert all(np.array_equal(a, b) for a, b in zip(*(s.stats(count, first) for s in stores)))
    for s in stores:
        got = s.stats(count, first)
        for i, r in enumerate(rows):
            sx, sxx = O.pattern_sums(r.cpu().numpy())
            assert got[0][i] == pytest.approx(sx, rel=1e-9, abs=1e-9) and got[1][i] == pytest.approx(sxx, rel=1e-10)
            assert got[2][i] == r.abs().max().item()
        s.close()


def busiest_xcd(T, ks, S):
    """Items of the XCD with the most, ids dealt to 8 in turn (the split item's after the others')."""
    whole, groups = (T - 1, -(-S // ks)) if ks > 1 else (T, 0)
    return whole * -(-S // 8) + -(-groups // 8)


@pytest.mark.parametrize("fmt,n", [("fp16", 786432), ("fp16", 2000000), ("split_bf16", 262144), ("fp8", 3145728),
                                   ("fp32", 2000000)])
@pytest.mark.parametrize("count,T,ks", [(300, 2, 2), (380, 2, 2), (120, 1, 4), (500, 3, 1)])
def test_split_items_shorten_the_launch(fmt, n, count, T, ks):
    """The slab of a plan: rounds of the busiest XCD's 32 CUs times the slab and
    the cost of one (24 stages, 2 for FP32) are not above those of the slab that
    items of one slab at a time would get."""
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    values = {"split_bf16": 32, "fp32": 32, "fp16": 64, "fp8": 128}[fmt]
    blocks, extra = -(-n // values), 2 if fmt == "fp32" else 24
    gram = csi.GramNCC(n // 2, 2)
    store = csi.PatternStore(n, count, fmt)
    plan = csi.GramPlan(gram, [(store, 0, count)])
    info = plan.info()
    plan.close()
    store.close()
    gram.close()
    kcb = info["slab_values"] // values
    S = -(-blocks // kcb)
    split = info["work_items"] < T * S
    assert info["work_items"] == (T * S if not split else (T - 1) * S + -(-S // ks))
    steps = [16 + 8 * i for i in range(30)] + [256 + 32 * i for i in range(56)] + [2048 + 256 * i for i in range(600)]
    one = min((k for k in steps if k <= blocks), key=lambda k: (-(-(T * -(-blocks // k)) // 256) * (k + 2), k))
    cost = lambda T, ks, k: -(-busiest_xcd(T, ks, -(-blocks // k)) // 32) * (k + extra)  # noqa: E731
    assert kcb <= one and cost(T, ks if split else 1, kcb) <= cost(T, 1, one)
    if ks == 1:
        assert kcb == one
