"""What this package is timed on: the calls of a common-source identification job.

A job decodes camera frames (``decode``), turns each into its PRNU pattern or
spectrum (``extract``), and compares patterns: one pair at a time (``pair``),
all pairs of a set (``compare`` through a pattern store, ``gram`` over separate
buffers, ``groups`` for cameras of several resolutions, ``pce`` from spectra),
or a few queries against a fingerprint store (``query``).  Sizes are those of
this package's configurations (512x512, 1024x1024, 2048x1536 and 4000x3000
frames); drawn cases spread over the sizes between and around them.
"""
import math

import numpy as np
import torch

from rocket_amd import _lib, csi, jpeg, serving

FORMATS = {"rgb8": (_lib.INPUT_RGB8, 3), "gray8": (_lib.INPUT_GRAY8, 1), "float32": (_lib.INPUT_FLOAT32, 1)}
VARIANTS = {"reference": _lib.PCE_REFERENCE, "textbook": _lib.PCE_TEXTBOOK}


def listed():
    return [
        # one small frame through the per-image call: what an interactive tool waits for
        {"name": "extract one 512x512 gray", "kind": "extract", "h": 512, "w": 512, "batch": 1, "format": "gray8",
         "spectrum": False},
        # a batch of ordinary camera frames into NCC patterns: the ingest of a large set
        {"name": "extract 32 of 2048x1536 rgb", "kind": "extract", "h": 1536, "w": 2048, "batch": 32,
         "format": "rgb8", "spectrum": False},
        # a batch of cropped frames into spectra: the ingest of a PCE job
        {"name": "extract 16 of 1024x1024 spectra", "kind": "extract", "h": 1024, "w": 1024, "batch": 16,
         "format": "rgb8", "spectrum": True},
        # full camera resolution, sides that are no powers of two
        {"name": "extract 4 of 4000x3000 rgb", "kind": "extract", "h": 3000, "w": 4000, "batch": 4, "format": "rgb8",
         "spectrum": False},
        # every pair of a set of spectra, reference scores
        {"name": "pce all pairs 40 of 1024x1024", "kind": "pce", "h": 1024, "w": 1024, "count": 40,
         "variant": "reference"},
        # every pair of a small set of larger frames, textbook scores
        {"name": "pce all pairs 12 of 2048x1536", "kind": "pce", "h": 1536, "w": 2048, "count": 12,
         "variant": "textbook"},
        # one pair of patterns through the drop-in call
        {"name": "ncc one pair 2048x1536", "kind": "pair", "h": 1536, "w": 2048, "strategy": "NCC"},
        # patterns into a store, then every pair of the set: the headline comparison
        {"name": "compare 1024 of 2048x1536", "kind": "compare", "h": 1536, "w": 2048, "count": 1024,
         "precision": "split_bf16"},
        # a ragged count of patterns in buffers of their own, FP32 products
        {"name": "gram 300 of 640x480 fp32", "kind": "gram", "h": 480, "w": 640, "count": 300, "precision": "fp32"},
        # cameras of three resolutions compared in one launch, half-size stores
        {"name": "groups 500 300 120 fp16", "kind": "groups", "counts": "500,300,120", "sizes": "1024x1024,2048x1536,4000x3000",
         "precision": "fp16"},
        # a small batch of queries against a few thousand cameras
        {"name": "query 8 of 4000 at 1024x1024", "kind": "query", "h": 1024, "w": 1024, "count": 4000, "queries": 8,
         "k": 10},
        # files as a camera writes them, from host memory to RGB8 on the device
        {"name": "decode 16 of 2048x1536", "kind": "decode", "h": 1536, "w": 2048, "count": 16, "step": 2},
    ]


def _side(rng, lo, hi):
    """A length 2^a 3^b 5^c between lo and hi, spread over the logarithm."""
    smooth = [v for v in (2 ** a * 3 ** b * 5 ** c for a in range(13) for b in range(8) for c in range(6))
              if lo <= v <= hi]
    at = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(smooth, key=lambda v: abs(math.log(v / at)))


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["extract", "extract", "extract", "pce", "pce", "pair", "compare", "gram", "groups", "query",
                       "decode"])
    if kind == "decode":
        h, w = rng.randrange(240, 2400), rng.randrange(320, 3200)
        return {"kind": kind, "h": h, "w": w, "count": min(_log_int(rng, 1, 32), max(1, 50_000_000 // (h * w))),
                "step": rng.choice([2, 4, 8])}
    if kind == "query":
        h, w = _side(rng, 256, 1024), _side(rng, 256, 1024)
        return {"kind": kind, "h": h, "w": w, "count": _log_int(rng, 100, 4000), "queries": _log_int(rng, 1, 64),
                "k": rng.choice([1, 5, 10])}
    if kind == "groups":
        sides = [(_side(rng, 200, 2000), _side(rng, 200, 2000)) for _ in range(rng.choice([2, 3, 4]))]
        return {"kind": kind, "sizes": ",".join("%dx%d" % s for s in sides),
                "counts": ",".join(str(_log_int(rng, 20, 500)) for _ in sides),
                "precision": rng.choice(["split_bf16", "fp16", "fp8"])}
    h, w = _side(rng, 45, 4000), _side(rng, 45, 4000)
    if kind == "extract":
        most = max(1, min(32, 100_000_000 // (h * w)))
        return {"kind": kind, "h": h, "w": w, "batch": rng.choice([1, _log_int(rng, 1, most)]),
                "format": rng.choice(["rgb8", "rgb8", "gray8", "float32"]), "spectrum": rng.random() < 0.35}
    if kind == "pce":
        most = max(2, min(40, int(math.sqrt(2 * 400_000_000 / (h * w)))))
        return {"kind": kind, "h": h, "w": w, "count": _log_int(rng, 2, most),
                "variant": rng.choice(["reference", "textbook"])}
    if kind == "pair":
        return {"kind": kind, "h": h, "w": w, "strategy": rng.choice(["NCC", "NCC", "PCE"])}
    most = max(2, min(1024, 1_000_000_000 // (h * w)))
    return {"kind": kind, "h": h, "w": w, "count": _log_int(rng, 2, most),
            "precision": rng.choice(["split_bf16", "fp32", "fp8"] + (["fp16"] if kind == "compare" else []))}


# ------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _frames(case, seed, count, channels):
    """uint8 camera frames: a smooth scene, the camera's multiplicative
    fingerprint, and read noise of two levels."""
    h, w = case["h"], case["w"]
    g = _generator(seed)
    y = torch.arange(h, device="cuda", dtype=torch.float32)[:, None] / h
    x = torch.arange(w, device="cuda", dtype=torch.float32)[None, :] / w
    camera = 1 + 0.02 * torch.randn((h, w), generator=g, device="cuda")
    shape = (count, h, w, channels) if channels > 1 else (count, h, w)
    out = torch.empty(shape, dtype=torch.uint8, device="cuda")
    waves = torch.rand((count, 4, 3), generator=g, device="cuda").cpu().numpy()
    for i in range(count):
        scene = 128.0
        for a, b, p in waves[i]:
            scene = scene + 20 * torch.cos(2 * math.pi * (int(5 * a) * x + int(5 * b) * y + float(p)))
        scene = scene * camera
        if channels > 1:
            scene = scene[:, :, None] * torch.tensor([1.0, 0.9, 0.8], device="cuda")
        noise = torch.randn(shape[1:], generator=g, device="cuda")
        out[i] = (scene + 2 * noise).round().clamp(0, 255).to(torch.uint8)
    return out


def _images(case, seed):
    _, channels = FORMATS[case["format"]]
    img = _frames(case, seed, case["batch"], channels)
    return img.to(torch.float32) if case["format"] == "float32" else img


def _patterns(n, count, seed, cameras=8, first=0):
    """`count` zero-mean patterns of n values, pattern i with a share of
    camera (first + i) % cameras' fingerprint."""
    g = _generator(seed)
    prints = torch.randn((cameras, n), generator=g, device="cuda")
    g = _generator(seed + 7919 * (first + 1))
    out = torch.empty((count, n), device="cuda")
    for i in range(count):
        torch.randn(n, generator=g, out=out[i])
        out[i].add_(prints[(first + i) % cameras], alpha=0.1)
        out[i] -= out[i].mean()
    return out


def _spectra(case, seed, count):
    """Half spectra of `count` patterns, as PCE extraction leaves them."""
    h, w = case["h"], case["w"]
    out = torch.empty((count, h, w // 2 + 1, 2), device="cuda")
    pats = _patterns(h * w, count, seed, cameras=4)
    for i in range(count):
        out[i] = torch.view_as_real(torch.fft.rfft2(pats[i].view(h, w)))
    return out


def _groups(case):
    sizes = [tuple(int(v) for v in s.split("x")) for s in case["sizes"].split(",")]
    return [(a * b, int(c)) for (a, b), c in zip(sizes, case["counts"].split(","))]


QUERY_CHUNK = 250  # fingerprints enrolled at a time


def _query_patterns(case, seed):
    """Two query patterns in three come from enrolled cameras."""
    n, count = case["h"] * case["w"], case["count"]
    q = _patterns(n, case["queries"], seed + 1)
    for i in range(case["queries"]):
        if i % 3 < 2:
            slot = (37 * i + 11) % count
            q[i] += 0.3 * _enrolled(case, seed, slot // QUERY_CHUNK)[slot % QUERY_CHUNK]
    return q


def _enrolled(case, seed, chunk):
    first = chunk * QUERY_CHUNK
    f = torch.randn((min(QUERY_CHUNK, case["count"] - first), case["h"] * case["w"]),
                    generator=_generator(seed + 31 * (chunk + 1)), device="cuda")
    return f.sub_(f.mean(dim=1, keepdim=True))


# ------------------------------------------------- JPEG files of the frames
_ZIGZAG = sorted(range(64), key=lambda p: (p // 8 + p % 8, p // 8 if (p // 8 + p % 8) % 2 else p % 8))
# the JPEG standard's example tables: (bits, values) for luminance and chrominance
_DC = [([0, 1, 5, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0, 0, 0], list(range(12))),
       ([0, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0, 0], list(range(12)))]
_AC = [([0, 2, 1, 3, 3, 2, 4, 3, 5, 5, 4, 4, 0, 0, 1, 125],
        list(bytes.fromhex("01020300041105122131410613516107227114328191a1082342b1c11552d1f02433627282"))),
       ([0, 2, 1, 2, 4, 4, 3, 4, 7, 5, 4, 4, 0, 1, 2, 119],
        list(bytes.fromhex("0001020311040521310612415107617113223281081442"
                           "91a1b1c109233352f0156272d10a162434e125f1")))]
for _, _vals in _AC:  # the longest codes: the remaining symbols in order
    _vals += [r * 16 + s for r in range(16) for s in range(1, 11) if r * 16 + s not in _vals]


def _codes(bits, vals):
    """(code, length) of every symbol of a canonical Huffman table."""
    code, at = 0, 0
    table = np.zeros((256, 2), dtype=np.int64)
    for length, many in enumerate(bits, 1):
        for _ in range(many):
            table[vals[at]] = code, length
            code, at = code + 1, at + 1
        code <<= 1
    return torch.from_numpy(table).cuda()


def _bit_length(v):
    return torch.ceil(torch.log2(v.abs().to(torch.float64) + 1)).to(torch.int64)


def _encode(rgb, step):
    """A baseline 4:2:0 JPEG file of an (h, w, 3) uint8 CUDA tensor."""
    h, w = int(rgb.shape[0]), int(rgb.shape[1])
    f = rgb.to(torch.float32).permute(2, 0, 1)[None]
    f = torch.nn.functional.pad(f, (0, -w % 16, 0, -h % 16), mode="replicate")[0]
    y = 0.299 * f[0] + 0.587 * f[1] + 0.114 * f[2]
    chroma = torch.stack([0.564 * (f[2] - y), 0.713 * (f[0] - y)])
    chroma = chroma.view(2, y.shape[0] // 2, 2, y.shape[1] // 2, 2).mean(dim=(2, 4))
    my, mx = y.shape[0] // 16, y.shape[1] // 16
    k = np.arange(8)
    dct = np.sqrt(0.25) * np.cos((2 * k[None, :] + 1) * k[:, None] * np.pi / 16)
    dct[0] /= np.sqrt(2)
    both = torch.from_numpy(np.kron(dct, dct)[_ZIGZAG]).to("cuda", torch.float32)   # 64 x 64, zigzag rows
    quant = np.array([min(255, step + step * (p // 8 + p % 8) // 2) for p in _ZIGZAG], dtype=np.uint8)
    luma = (y - 128).view(my, 2, 8, mx, 2, 8).permute(0, 3, 1, 4, 2, 5).reshape(my * mx, 4, 64)
    chroma = chroma.view(2, my, 8, mx, 8).permute(1, 3, 0, 2, 4).reshape(my * mx, 2, 64)
    blocks = torch.cat([luma, chroma], dim=1)                                       # MCU order
    coef = (blocks @ both.T / torch.from_numpy(quant).cuda()).round().to(torch.int64)
    coef = coef.clamp(-1023, 1023)
    dc = coef[:, :, 0].clone()
    flat = dc[:, :4].reshape(-1)
    dc[:, :4] = torch.diff(flat, prepend=flat[:1] * 0).view(-1, 4)
    dc[:, 4:] = torch.diff(dc[:, 4:], dim=0, prepend=dc[:1, 4:] * 0)
    v = coef.reshape(-1, 64)
    v[:, 0] = dc.reshape(-1)
    # one slot per coefficient (its zero-run codes, code and extra bits) and one for the end of block
    size = _bit_length(v)
    extra = torch.where(v < 0, v + (1 << size) - 1, v)
    dc_codes, ac_codes = (torch.stack([_codes(*t) for t in tables]) for tables in (_DC, _AC))
    table = (torch.arange(6, device="cuda") // 4).repeat(v.shape[0] // 6)           # of each block
    place = torch.arange(64, device="cuda").expand_as(v)
    last = torch.cummax(torch.where((v != 0) | (place == 0), place, 0), dim=1).values
    run = place - torch.cat([last[:, :1], last[:, :-1]], dim=1) - 1
    run[:, 0] = 0
    code, length = ac_codes[table[:, None], (run % 16) * 16 + size].unbind(-1)
    code[:, 0], length[:, 0] = dc_codes[table, size[:, 0]].unbind(-1)
    value, bits = (code << size) | extra, length + size
    zrl, zrl_bits = ac_codes[table, 0xF0][:, None].unbind(-1)
    for many in (1, 2, 3):
        value = torch.where(run // 16 >= many, value + (zrl << (bits + (many - 1) * zrl_bits)), value)
    bits = bits + (run // 16) * zrl_bits
    bits = torch.where((v != 0) | (place == 0), bits, 0)
    end = ac_codes[table, 0]
    value = torch.cat([value, end[:, :1]], dim=1).reshape(-1)
    bits = torch.cat([bits, torch.where(last[:, 63:] < 63, end[:, 1:], 0)], dim=1).reshape(-1)
    value, bits = value[bits > 0], bits[bits > 0]
    until = torch.cumsum(bits, 0)
    total = int(until[-1])
    which = torch.repeat_interleave(torch.arange(len(bits), device="cuda"), bits)
    stream = (value[which] >> (until[which] - 1 - torch.arange(total, device="cuda"))) & 1
    stream = torch.cat([stream, torch.ones(-total % 8, dtype=torch.int64, device="cuda")]).view(-1, 8)
    scan = (stream << torch.arange(7, -1, -1, device="cuda")).sum(1)
    wide = torch.repeat_interleave(scan, 1 + (scan == 255).to(torch.int64))         # a zero after each 255
    stuffed = torch.cumsum(1 + (scan == 255).to(torch.int64), 0)[scan == 255] - 1
    wide[stuffed] = 0
    head = b"\xff\xd8\xff\xdb\x00\x43\x00" + quant.tobytes()
    head += b"\xff\xc0\x00\x11\x08" + h.to_bytes(2, "big") + w.to_bytes(2, "big") + bytes([3, 1, 34, 0, 2, 17, 0, 3, 17, 0])
    for kind, tables in ((0, _DC), (16, _AC)):
        for k, (counts, vals) in enumerate(tables):
            head += b"\xff\xc4" + (19 + len(vals)).to_bytes(2, "big") + bytes([kind + k]) + bytes(counts) + bytes(vals)
    head += bytes([255, 218, 0, 12, 3, 1, 0, 2, 17, 3, 17, 0, 63, 0])
    return head + wide.to(torch.uint8).cpu().numpy().tobytes() + b"\xff\xd9"


# ---------------------------------------------------------------- the cases
def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "extract":
        h, w = case["h"], case["w"]
        s["filter"] = csi.PRNUFilter(h, w, apply_spectral_filter=case["spectrum"])
        s["images"] = _images(case, seed).view(case["batch"], -1)
        s["out"] = torch.empty((case["batch"], s["filter"].get_output_size() // 4), device="cuda")
    elif kind == "pce":
        s["cmp"] = csi.PeakToCorrelationEnergy(case["h"], case["w"], VARIANTS[case["variant"]])
        s["spectra"] = _spectra(case, seed, case["count"])
        s["pairs"] = np.array([(i, j) for i in range(case["count"]) for j in range(i + 1, case["count"])],
                              dtype=np.int32)
    elif kind == "pair":
        s["ctx"] = csi.CommonSourceIdentificationContext(case["h"], case["w"],
                                                         csi.ComparisonStrategy[case["strategy"]])
        s["pair"] = (_spectra(case, seed, 2) if case["strategy"] == "PCE"
                     else _patterns(case["h"] * case["w"], 2, seed, cameras=1))
        s["out"] = torch.empty(1, dtype=torch.float64, device="cuda")
    elif kind in ("compare", "gram"):
        n, count = case["h"] * case["w"], case["count"]
        s["gram"] = csi.GramNCC(case["h"], case["w"])
        s["patterns"] = _patterns(n, count, seed, cameras=16)
        if kind == "compare":
            s["store"] = csi.PatternStore(n, count, case["precision"])
        s["out"] = torch.empty((count, count), dtype=torch.float64, device="cuda")
    elif kind == "groups":
        s["gram"] = csi.GramNCC(64, 64)
        s["stores"] = []
        for g, (n, count) in enumerate(_groups(case)):
            store = csi.PatternStore(n, count, case["precision"])
            store.put(_patterns(n, count, seed + g))
            s["stores"].append(store)
        s["plan"] = csi.GramPlan(s["gram"], [(t, 0, t.capacity) for t in s["stores"]])
    elif kind == "query":
        s["ctx"] = csi.CommonSourceIdentificationContext(case["h"], case["w"])
        s["store"] = serving.FingerprintStore(case["h"], case["w"], case["count"])
        for chunk in range(-(-case["count"] // QUERY_CHUNK)):
            s["store"].put(_enrolled(case, seed, chunk), first_slot=chunk * QUERY_CHUNK)
        s["queries"] = _query_patterns(case, seed)
    else:
        s["decoder"] = jpeg.JpegDecoder()
        s["files"] = [_encode(f, case["step"]) for f in _frames(case, seed, case["count"], 3)]
        s["out"] = torch.empty((case["count"], case["h"], case["w"], 3), dtype=torch.uint8, device="cuda")
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "extract":
        fmt = FORMATS[case["format"]][0]
        if case["batch"] == 1:
            s["filter"].apply_gpu(s["images"], s["out"], fmt)
        else:
            s["filter"].apply_gpu_batch(s["images"], s["out"], fmt)
        return s["out"]
    if kind == "pce":
        return s["cmp"].pairs(s["spectra"], s["pairs"])
    if kind == "pair":
        s["ctx"].correlate_gpu("a", s["pair"][0], "b", s["pair"][1], s["out"])
        return s["out"]
    if kind == "compare":
        s["store"].put(s["patterns"], sync=False)
        return s["store"].gram(s["gram"], case["count"], out=s["out"])
    if kind == "gram":
        return s["gram"].ncc(s["patterns"], case["precision"], out=s["out"])
    if kind == "groups":
        return s["plan"].run()
    if kind == "query":
        return s["store"].query(s["ctx"]._ctx, s["queries"], k=case["k"])
    return s["decoder"].decode(s["files"], out=s["out"])


def work(case):
    kind = case["kind"]
    if kind == "groups":
        groups = _groups(case)
        width = {"fp32": 4, "split_bf16": 4, "fp16": 2, "fp8": 1}[case["precision"]]
        return {"bytes": sum(width * n * c + 8 * c * c for n, c in groups), "flops": sum(c * (c + 1) * n for n, c in groups)}
    h, w = case["h"], case["w"]
    n, half = h * w, h * (w // 2 + 1)
    fft = 2.5 * n * math.log2(n)  # of real data
    if kind == "extract":
        pixel = {"rgb8": 3, "gray8": 1, "float32": 4}[case["format"]]
        return {"bytes": case["batch"] * (pixel * n + (8 * half if case["spectrum"] else 4 * n)),
                "flops": case["batch"] * ((3 if case["spectrum"] else 2) * fft + 60 * n)}
    if kind == "pce":
        c = case["count"]
        return {"bytes": 8 * half * c + 8 * c * (c - 1), "flops": c * (c - 1) // 2 * (fft + 12 * n)}
    if kind == "pair":
        if case["strategy"] == "PCE":
            return {"bytes": 16 * half + 8, "flops": fft + 12 * n}
        return {"bytes": 8 * n + 8, "flops": 10 * n}
    if kind in ("compare", "gram"):
        c = case["count"]
        return {"bytes": 4 * n * c + 8 * c * c, "flops": c * (c + 1) * n}
    if kind == "query":
        q = case["queries"]
        return {"bytes": n * case["count"] + 4 * n * q * (1 + case["k"]), "flops": 2 * n * case["count"] * q}
    return {"bytes": case["count"] * 3.15 * n, "flops": case["count"] * 40 * n}


# ------------------------------------------------- the same numbers in 64 bits
def _gradient(a, dim):
    d = torch.empty_like(a)
    size = a.shape[dim]
    mid = 0.5 * (a.narrow(dim, 2, size - 2) - a.narrow(dim, 0, size - 2)) if size > 2 else None
    if mid is not None:
        d.narrow(dim, 1, size - 2).copy_(mid)
    d.narrow(dim, 0, 1).copy_(a.narrow(dim, 1, 1) - a.narrow(dim, 0, 1))
    d.narrow(dim, size - 1, 1).copy_(a.narrow(dim, size - 1, 1) - a.narrow(dim, size - 2, 1))
    return d


def _zero_mean_rows(x):
    x = x.clone()
    x[0::2] -= x[0::2].mean(dim=0, keepdim=True)
    x[1::2] -= x[1::2].mean(dim=0, keepdim=True)
    return x


def _exact_pattern(img, channels):
    """Gray, first-step total variation, zero mean per parity, Wiener filter."""
    weight = [float(np.float32(v)) for v in (0.299, 0.587, 0.114)]
    img = img.to(torch.float64)
    if channels == 3:
        gray = weight[0] * img[..., 2] + weight[1] * img[..., 1] + weight[2] * img[..., 0]
    else:
        gray = img * (sum(weight) if channels == 1 else 1.0)
    dx, dy = _gradient(gray, 1), _gradient(gray, 0)
    scale = 1 / (1 + torch.sqrt(dx * dx + dy * dy))
    x = _gradient(dx * scale, 1) + _gradient(dy * scale, 0)
    x = _zero_mean_rows(_zero_mean_rows(x).T).T
    f = torch.fft.fft2(x)
    power = (f.real * f.real + f.imag * f.imag)[None, None]
    least = None
    for size in (3, 5, 7, 9):
        box = torch.nn.functional.avg_pool2d(power, size, stride=1, padding=size // 2)
        least = box if least is None else torch.minimum(least, box)
    n = x.numel()
    var = (x * x).sum() * n / (n - 1)
    f = f * (var / torch.maximum(var, least[0, 0]))
    return torch.fft.ifft2(f).real


def _exact_pce(x, y, h, w, variant):
    x, y = x.to(torch.complex128), y.to(torch.complex128)
    half = w // 2 + 1
    if variant == "textbook":
        c = torch.fft.irfft2(x.conj() * y, s=(h, w))
    else:  # the right half mirrored from the same row
        full = torch.empty((h, w), dtype=torch.complex128, device=x.device)
        full[:, :half] = x.conj() * y
        at = w - torch.arange(half, w, device=x.device)
        full[:, half:] = x[:, at] * y[:, at].conj()
        c = torch.fft.ifft2(full).real
    py, px = divmod(int(c.abs().argmax()), w)
    rows, cols = torch.arange(h, device=x.device), torch.arange(w, device=x.device)
    if variant == "textbook":
        inside = ((((rows - py + 5) % h) < 11)[:, None]) & ((((cols - px + 5) % w) < 11)[None, :])
        peak, outside = c[py, px], h * w - int(inside.sum())
    else:
        inside = ((rows - py).abs() < 5)[:, None] & ((cols - px).abs() < 5)[None, :]
        peak, outside = c[h - 1, w - 1], h * w - 121
    energy = (c * c).masked_fill(inside, 0).sum() / outside
    return (torch.sign(peak) if variant == "textbook" else 1) * peak * peak / energy


def _exact_ncc(p):
    """NCC matrix of float32 rows: products and sums in 64 bits."""
    count, n = p.shape
    g = torch.zeros((count, count), dtype=torch.float64, device=p.device)
    s = torch.zeros(count, dtype=torch.float64, device=p.device)
    for k in range(0, n, 1 << 19):
        part = p[:, k:k + (1 << 19)].to(torch.float64)
        g += part @ part.T
        s += part.sum(dim=1)
    d = torch.sqrt(torch.diagonal(g) - s * s)
    return g / (d[:, None] * d[None, :])


def exact(case, seed):
    kind = case["kind"]
    if kind == "extract":
        channels = {"rgb8": 3, "gray8": 1, "float32": 0}[case["format"]]
        out = []
        for img in _images(case, seed):
            x = _exact_pattern(img, channels)
            out.append(torch.view_as_real(torch.fft.rfft2(x)).reshape(-1) if case["spectrum"] else x.reshape(-1))
        return torch.stack(out)
    if kind == "pce":
        sp = torch.view_as_complex(_spectra(case, seed, case["count"]))
        return torch.stack([_exact_pce(sp[i], sp[j], case["h"], case["w"], case["variant"])
                            for i in range(case["count"]) for j in range(i + 1, case["count"])])
    if kind == "pair":
        if case["strategy"] == "PCE":
            a, b = torch.view_as_complex(_spectra(case, seed, 2))
            return _exact_pce(a, b, case["h"], case["w"], "reference").reshape(1)
        return _exact_ncc(_patterns(case["h"] * case["w"], 2, seed, cameras=1))[0, 1].reshape(1)
    if kind in ("compare", "gram"):
        return _exact_ncc(_patterns(case["h"] * case["w"], case["count"], seed, cameras=16))
    if kind == "groups":
        return [_exact_ncc(_patterns(n, count, seed + g)) for g, (n, count) in enumerate(_groups(case))]
    if kind == "query":  # the true best scores; which fingerprints they are is whole numbers
        q = _query_patterns(case, seed).to(torch.float64)
        best = []
        for chunk in range(-(-case["count"] // QUERY_CHUNK)):
            f = _enrolled(case, seed, chunk).to(torch.float64)
            d = torch.sqrt((f * f).sum(1) - f.sum(1) ** 2)
            best.append(q @ f.T / d[None, :])
        score = torch.cat(best, dim=1) / torch.sqrt((q * q).sum(1) - q.sum(1) ** 2)[:, None]
        return None, torch.sort(score, dim=1, descending=True).values[:, :case["k"]]
    return None
