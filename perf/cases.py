"""Performance cases of the codec: what a user's program has it do, over the range of sizes in use.

A case is a dict of plain values:

* ``op``: ``compress`` / ``decompress`` (uint16), ``compress_u32`` / ``decompress_u32``, ``batch_compress`` /
  ``batch_decompress`` (many frames, one plan) or ``quality`` (error metrics of a lossy round trip);
* ``x, y, z``: frames, rows and columns of the volume (``x`` = number of frames of a batch, whose sides are
  drawn from ``mix``);
* ``kind``: what the detector saw -- ``sparse`` (Poisson 0.05 and hot pixels), ``cssi`` (Poisson 0.3, Bragg peaks
  of up to ``amp`` counts, gap stripes), ``xpcs`` (speckle, ``amp`` / 1000 counts a pixel on average) or ``dense``
  (tomography: a smooth object of up to ``amp`` counts with noise);
* ``b0 .. b3, pooling``: the setting; lossless is 1 1 1 1 and 1;
* ``blocking``: the call returns with the size or status on the host, else it is stream-ordered.

Volumes and streams live in device memory, as the entry points take them, and a program that compresses frame
after frame keeps its output buffers; inputs are drawn on the GPU from the seed.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("sc25-lscomp_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import lscomp  # noqa: E402

LOSSLESS = (1, 1, 1, 1, 1.0)
# settings in use beside lossless: the four-bin one and the equal-bin ones of the benchmark, and the XPCS ones
LOSSY = ((3, 5, 10, 15, 0.5), (3, 3, 3, 3, 0.5), (5, 5, 5, 5, 0.5), (10, 10, 10, 10, 0.5), (3, 4, 5, 6, 0.7),
         (10, 11, 12, 13, 0.7))
SIDES = (256, 512, 768, 1024, 1536, 2048)   # frame sides of a batch


def _case(name, op, x, y, z, kind, setting, blocking, amp=60000):
    b0, b1, b2, b3, p = setting
    return {"name": name, "op": op, "x": x, "y": y, "z": z, "kind": kind, "b0": b0, "b1": b1, "b2": b2, "b3": b3,
            "pooling": p, "blocking": blocking, "amp": amp}


def listed():
    lossy4, b3 = LOSSY[0], LOSSY[1]
    return [
        # one small frame between two readouts: the time of a call
        _case("frame512_compress", "compress", 1, 512, 512, "sparse", LOSSLESS, True),
        # a short series looked at again: a small stored stream read back
        _case("series16_decompress", "decompress", 16, 512, 512, "sparse", LOSSLESS, True),
        # one large frame of a lossy live stream, queued without waiting for its size
        _case("frame2048_compress_lossy", "compress", 1, 2048, 2048, "cssi", lossy4, False),
        # a whole scan (the headline volume): stored losslessly, read back, and its lossy stream read back
        _case("cssi_compress", "compress", 600, 1813, 1558, "cssi", LOSSLESS, True),
        _case("cssi_decompress", "decompress", 600, 1813, 1558, "cssi", LOSSLESS, False),
        _case("cssi_decompress_lossy", "decompress", 600, 1813, 1558, "cssi", lossy4, True),
        # a speckle series, rows at 16-byte boundaries, lossy
        _case("xpcs_compress_lossy", "compress", 512, 1024, 1024, "xpcs", b3, True, 300),
        # tomography, which hardly compresses: odd sides going in, even ones coming back
        _case("dense_odd_compress", "compress", 800, 621, 621, "dense", LOSSLESS, True, 1500),
        _case("dense_decompress", "decompress", 750, 1024, 1024, "dense", LOSSLESS, True, 3000),
        # 32-bit counts of half a scan
        _case("u32_compress", "compress_u32", 300, 1813, 1558, "cssi", LOSSLESS, True, 1 << 22),
        # frames of several detectors in one launch
        dict(_case("batch_compress", "batch_compress", 512, 0, 0, "xpcs", LOSSLESS, True, 20), mix=4),
        # what a lossy setting costs: PSNR family and SSIM of a speckle series
        _case("quality_xpcs", "quality", 512, 1024, 1024, "xpcs", b3, True, 300),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(("compress",) * 4 + ("decompress",) * 4 + ("compress_u32", "decompress_u32", "batch_compress",
                                                             "batch_decompress", "quality"))
    setting = LOSSLESS if rng.random() < 0.5 else rng.choice(LOSSY)
    if op == "quality":
        setting = rng.choice(LOSSY)
    if op.startswith("batch"):
        kind = rng.choice(("xpcs", "cssi"))
        amp = _log_int(rng, 20, 500) if kind == "xpcs" else 60000
        return {k: v for k, v in dict(_case("", op, _log_int(rng, 16, 512), 0, 0, kind, setting, True, amp),
                                      mix=rng.randrange(1 << 20)).items() if k != "name"}
    kind = rng.choice(("sparse", "cssi", "xpcs", "dense"))
    u32 = op.endswith("u32")
    # largest volumes: the headline volume's bytes (half for dense ones, whose streams are as large); the metrics'
    # listed volume
    most = 512 * 1024 * 1024 if op == "quality" else 600 * 1813 * 1558 // ((1 + u32) * (1 + (kind == "dense")))
    n = _log_int(rng, 1 << 18, most)
    y, z = _log_int(rng, 185, 2167), _log_int(rng, 185, 2167)
    lo = 16 if op == "quality" else 1
    x = max(lo, min(n // (y * z), most // (y * z)))
    amp = _log_int(rng, 200, 30000) if kind == "dense" else _log_int(rng, 20, 500) if kind == "xpcs" else \
        1 << 22 if u32 else 60000
    blocking = op == "quality" or x * y * z > 1 << 26 or rng.random() < 0.5
    return {k: v for k, v in _case("", op, x, y, z, kind, setting, blocking, amp).items() if k != "name"}


# ---- inputs -----------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _frames_per_step(y, z):
    return max(1, (1 << 26) // (y * z))


def _exponential(shape, g):
    return torch.empty(shape, device="cuda").exponential_(generator=g)


def _add_peaks(v, amp, g):
    """50 Gaussian peaks per frame, sigma 1..3 pixels, up to amp counts, added to int32 frames."""
    f, y, z = v.shape
    u = torch.rand((4, f, 50), generator=g, device="cuda")
    cy, cz, sigma, a = u[0] * y, u[1] * z, 1 + 2 * u[2], 100 + (amp - 100) * u[3]
    o = torch.arange(-12, 13, device="cuda")
    yy = cy.floor().long()[..., None] + o
    zz = cz.floor().long()[..., None] + o
    s2 = (2 * sigma * sigma)[..., None]
    gy = torch.exp(-(yy + 0.5 - cy[..., None]) ** 2 / s2) * ((yy >= 0) & (yy < y))
    gz = torch.exp(-(zz + 0.5 - cz[..., None]) ** 2 / s2) * ((zz >= 0) & (zz < z))
    w = (a[..., None, None] * gy[..., :, None] * gz[..., None, :] + 0.5).to(torch.int32)
    at = (torch.arange(f, device="cuda")[:, None, None, None] * y + yy.clamp(0, y - 1)[..., :, None]) * z \
        + zz.clamp(0, z - 1)[..., None, :]
    v.view(-1).index_add_(0, at.reshape(-1), w.reshape(-1))


def _fill(out, kind, amp, seed):
    """Fills an int16- or int32-typed (x, y, z) volume (unsigned bits) with detector counts."""
    g = _generator(seed)
    x, y, z = out.shape
    top = 65535 if out.element_size() == 2 else (1 << 30)
    rate = None
    if kind == "xpcs":   # one speckle pattern, Poisson counts per frame
        rate = _exponential((y, z), g) * (amp / 1000) * sum(_exponential((y, z), g) for _ in range(4)) / 4
    elif kind == "dense":   # one smooth object, its projections, shot noise
        r = torch.linspace(-1, 1, y, device="cuda")[:, None] ** 2 + torch.linspace(-1, 1, z, device="cuda")[None] ** 2
        coarse = torch.rand((1, 1, 9, 9), generator=g, device="cuda")
        tex = torch.nn.functional.interpolate(coarse, size=(y, z), mode="bilinear", align_corners=True)[0, 0]
        rate = amp * (0.15 + 0.7 * torch.exp(-r) * (0.5 + 0.5 * tex))
    step = _frames_per_step(y, z)
    for f0 in range(0, x, step):
        f = min(step, x - f0)
        if kind == "dense":
            turn = 1 + 0.1 * torch.cos(torch.arange(f0, f0 + f, device="cuda") * 0.05)[:, None, None]
            mean = rate[None] * turn
            v = mean + mean.sqrt() * torch.randn(mean.shape, generator=g, device="cuda")
            v = v.round().clamp_(0, top).to(torch.int32)
        else:
            lam = rate.expand(f, y, z).contiguous() if rate is not None else \
                torch.full((f, y, z), 0.05 if kind == "sparse" else 0.3, device="cuda")
            v = torch.poisson(lam, generator=g).to(torch.int32)
            if kind == "sparse":   # 0.1 % hot pixels
                hot = torch.rand(v.shape, generator=g, device="cuda")
                v = torch.where(hot < 0.001, 200 + (hot * 3.8e6).to(torch.int32), v)
            elif kind == "cssi":
                _add_peaks(v, amp, g)
                s0, s1 = (512, 1032) if z > 1040 else (z // 3 & ~7, 2 * z // 3 & ~7)
                v[:, :, s0:s0 + 8] = 0   # gaps between detector modules
                v[:, :, s1:s1 + 8] = 0
        v.clamp_(0, top)
        out[f0:f0 + f].copy_(v.to(out.dtype) if out.element_size() == 4 else ((v + 32768) % 65536 - 32768).to(out.dtype))
    return out


def _volume(case, seed):
    dtype = torch.int32 if case["op"].endswith("u32") else torch.int16
    return _fill(torch.empty((case["x"], case["y"], case["z"]), dtype=dtype, device="cuda"), case["kind"], case["amp"],
                 seed)


def _bins(case):
    return (case["b0"], case["b1"], case["b2"], case["b3"])


def _sides(case):
    return [int(s) for s in np.random.RandomState(case["mix"]).choice(SIDES, size=case["x"])]


def _unsigned(v):
    return v.to(torch.int32) & 0xFFFF


def _approximation(vol, bin_):
    """What a decoder of a one-bin setting gives back: pairs averaged in the quiet blocks, counts rounded down."""
    out = torch.empty_like(vol)
    step = _frames_per_step(*vol.shape[1:])
    for f in range(0, vol.shape[0], step):
        v = _unsigned(vol[f:f + step])
        even = v.shape[2] // 2 * 2
        a, b = v[..., 0:even:2], v[..., 1:even:2]
        mean = torch.where((a < 64) & (b < 64), (a + b) // 2, a)
        v[..., 0:even:2] = mean
        v[..., 1:even:2] = torch.where((a < 64) & (b < 64), mean, b)
        v = v // bin_ * bin_
        out[f:f + step].copy_(((v + 32768) % 65536 - 32768).to(torch.int16))
    return out


def _prepare_batch(case, seed):
    sides = _sides(case)
    frames, at = [], 0
    pixels = torch.empty(sum(s * s for s in sides), dtype=torch.int16, device="cuda")
    for i, s in enumerate(sides):
        frames.append(pixels[at:at + s * s].view(1, s, s))
        at += s * s
    for s in sorted(set(sides)):   # the frames of one detector size are one series
        mine = [f for f, t in zip(frames, sides) if t == s]
        series = _fill(torch.empty((len(mine), s, s), dtype=torch.int16, device="cuda"), case["kind"], case["amp"],
                       seed * 16 + SIDES.index(s))
        for f, v in zip(mine, series):
            f.copy_(v[None])
    dims = [(1, s, s) for s in sides]
    caps = [-(-lscomp.max_compressed_bytes(d) // 256) * 256 for d in dims]
    arena = torch.zeros(sum(caps), dtype=torch.uint8, device="cuda")
    starts = np.cumsum([0] + caps)
    streams = [arena[int(a):int(b)] for a, b in zip(starts[:-1], starts[1:])]
    blocks = sum(lscomp.num_blocks(d) for d in dims)
    plan = lscomp.Plan(lscomp.COMPRESS, len(dims), blocks)
    plan.set_items([(f, d, _bins(case), case["pooling"], s, s.numel()) for f, d, s in zip(frames, dims, streams)])
    state = {"op": case["op"], "pixels": pixels, "arena": arena, "plan": plan}
    if case["op"] == "batch_decompress":
        plan.launch()
        sizes = plan.sizes()
        plan.close()
        out = torch.zeros_like(pixels)
        at, back = 0, []
        for s in sides:
            back.append(out[at:at + s * s].view(1, s, s))
            at += s * s
        plan = lscomp.Plan(lscomp.DECOMPRESS, len(dims), blocks)
        plan.set_items([(f, d, _bins(case), case["pooling"], s, n) for f, d, s, n in zip(back, dims, streams, sizes)])
        state.update(pixels=out, plan=plan)
    torch.cuda.synchronize()
    return state


def prepare(case, seed):
    if case["op"].startswith("batch"):
        return _prepare_batch(case, seed)
    dims = (case["x"], case["y"], case["z"])
    vol = _volume(case, seed)
    if case["op"] == "quality":
        return {"op": "quality", "dims": dims, "vol": vol, "dec": _approximation(vol, case["b0"])}
    u32 = case["op"].endswith("u32")
    state = {"op": case["op"], "dims": dims, "bins": _bins(case), "pooling": case["pooling"],
             "blocking": case["blocking"]}
    cap = lscomp.max_compressed_bytes_u32(dims) if u32 else lscomp.max_compressed_bytes(dims)
    out = torch.zeros(cap, dtype=torch.uint8, device="cuda")
    if case["op"].startswith("compress"):
        state.update(vol=vol, out=out, size=torch.zeros(1, dtype=torch.int64, device="cuda"))
        return state
    _, n = (lscomp.compress_u32 if u32 else lscomp.compress)(vol, dims, _bins(case), case["pooling"], out=out)
    state.update(stream=out[:n].clone(), out=torch.zeros_like(vol))
    return state


# ---- one pass ---------------------------------------------------------------

def run(s):
    op = s["op"]
    if op == "quality":
        return {"error": lscomp.error_stats(s["vol"], s["dec"]), "ssim": lscomp.ssim(s["vol"], s["dec"], s["dims"])}
    if op == "batch_compress":
        s["plan"].launch(graph=True)
        return s["arena"], np.array(s["plan"].sizes())
    if op == "batch_decompress":
        s["plan"].launch(graph=True)
        return s["pixels"], s["plan"].status()
    u32 = op.endswith("u32")
    if op.startswith("compress"):
        if s["blocking"]:
            f = lscomp.compress_u32 if u32 else lscomp.compress
            out, n = f(s["vol"], s["dims"], s["bins"], s["pooling"], out=s["out"])
            return out, n
        f = lscomp.compress_u32_async if u32 else lscomp.compress_async
        f(s["vol"], s["dims"], s["bins"], s["pooling"], s["out"], s["size"])
        return s["out"], s["size"]
    n = s["stream"].numel()
    if s["blocking"]:
        return (lscomp.decompress_u32 if u32 else lscomp.decompress)(s["stream"], n, s["dims"], s["bins"], out=s["out"])
    f = lscomp.decompress_u32_async if u32 else lscomp.decompress_async
    f(s["stream"], n, s["dims"], s["bins"], s["out"])
    return s["out"]


# ---- what a pass cannot do without ------------------------------------------

def _payload_per_block(case):
    """Mean payload bytes of a block (64 values), as these inputs give it."""
    lossless = case["b0"] == 1
    if case["kind"] == "dense":
        planes = math.log2(max(2.0, case["amp"] * 0.6 / case["b3"])) + 0.5
        return 8 * planes - 3
    if not lossless:
        return {"sparse": 1.0, "cssi": 0.6, "xpcs": (case["amp"] / 500) ** 4}[case["kind"]]
    if case["kind"] == "xpcs":
        return 6 * (case["amp"] / 20) ** 0.4
    return {"sparse": 13.5, "cssi": 16.0}[case["kind"]]


def work(case):
    if case["op"].startswith("batch"):
        shapes = [(1, s, s) for s in _sides(case)]
    else:
        shapes = [(case["x"], case["y"], case["z"])]
    n = sum(x * y * z for x, y, z in shapes)
    esize = 4 if case["op"].endswith("u32") else 2
    if case["op"] == "quality":   # both volumes; per window of the SSIM about 60 operations
        x, y, z = shapes[0]
        windows = ((x - 7) // 2 + 1) * ((y - 7) // 2 + 1) * ((z - 7) // 2 + 1)
        return {"bytes": 2 * esize * n, "flops": 60 * windows}
    blocks = sum(x * ((y + 7) // 8) * ((z + 7) // 8) for x, y, z in shapes)
    return {"bytes": esize * n + blocks * (1 + _payload_per_block(case)), "flops": 0}


# ---- the metrics in 64 bits -------------------------------------------------

def _window_sums(t, f):
    """Sliding sums (or maxima) over 7 values at stride 2 along the three axes."""
    for axis in range(3):
        n = (t.shape[axis] - 7) // 2 + 1
        acc = None
        for k in range(7):
            part = t[(slice(None),) * axis + (slice(k, k + 2 * n - 1, 2),)]
            acc = part.clone() if acc is None else f(acc, part)
        t = acc
    return t


def _exact_ssim(vol, dec):
    x = vol.shape[0]
    windows = (x - 7) // 2 + 1
    step = max(1, (1 << 25) // (vol.shape[1] * vol.shape[2]))
    total, count = 0.0, 0
    for k in range(0, windows, step):
        k1 = min(windows, k + step)
        a, b = (_unsigned(v[2 * k:2 * (k1 - 1) + 7]).to(torch.int64) for v in (vol, dec))
        sx, sy, sxx, syy, sxy = (_window_sums(t, torch.add).double() for t in (a, b, a * a, b * b, a * b))
        span = _window_sums(a, torch.maximum).double() + _window_sums(-a, torch.maximum).double()
        span = torch.where(span == 0, torch.ones_like(span), span)
        c1, c2 = (0.01 * span) ** 2, (0.03 * span) ** 2
        mx, my = sx / 343, sy / 343
        vx, vy, cov = ((343 * p - q * r) / 343 ** 2 for p, q, r in ((sxx, sx, sx), (syy, sy, sy), (sxy, sx, sy)))
        dx, dy = vx.sqrt(), vy.sqrt()
        s = (2 * mx * my + c1) / (mx * mx + my * my + c1) * (2 * dx * dy + c2) / (vx + vy + c2) \
            * (cov + c2 / 2) / (dx * dy + c2 / 2)
        total += float(s.sum())
        count += s.numel()
    return total / count


def _exact_error(vol, dec):
    se = sd = 0
    me, rel, lo, hi = 0, 0.0, 65535, 0
    step = _frames_per_step(*vol.shape[1:])
    for f in range(0, vol.shape[0], step):
        a, d = _unsigned(vol[f:f + step]).to(torch.int64), _unsigned(dec[f:f + step]).to(torch.int64)
        e = (a - d).abs()
        se += int((e * e).sum())
        sd += int((d * d).sum())
        me, lo, hi = max(me, int(e.max())), min(lo, int(a.min())), max(hi, int(a.max()))
        rel = max(rel, float(torch.where(a > 0, e.double() / a.clamp(min=1), 0.0).max()))
    n = vol.numel()
    mse, span = se / n, float(hi - lo)
    return {"n": n, "max_abs_err": me, "min_orig": lo, "max_orig": hi, "sum_sq_err": se, "sum_sq_dec": sd,
            "max_rel_err": rel, "mse": mse, "range": span,
            "psnr": 20 * math.log10(span) - 10 * math.log10(mse) if mse > 0 and span > 0 else None,
            "norm_err": math.sqrt(se), "norm_err_norm": math.sqrt(se) / math.sqrt(sd) if sd else None,
            "nrmse": math.sqrt(mse) / span if span else None}


def exact(case, seed):
    """The metrics; streams and decoded volumes are whole numbers."""
    if case["op"] != "quality":
        return None
    vol = _volume(case, seed)
    dec = _approximation(vol, case["b0"])
    return {"error": _exact_error(vol, dec), "ssim": _exact_ssim(vol, dec)}
