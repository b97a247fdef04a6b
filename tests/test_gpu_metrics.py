"""GPU error metrics against a float64 numpy restatement of the reference's
computePSNR definitions (lsCOMP/src/cuLSZ_utility.cu:887-946)."""
import numpy as np
import pytest

from lsc_helpers import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,offset", [(1, 0), (7, 0), (4096, 0), (1000003, 0), (1000003, 1)])
def test_metrics_vs_numpy(gpu, n, offset):
    import torch
    rng = np.random.default_rng(n)
    a = rng.integers(0, 65536, n + 1).astype(np.uint16)[offset:offset + n]
    d = np.clip(a.astype(np.int64) + rng.integers(-40, 41, n), 0, 65535).astype(np.uint16)
    ta = torch.from_numpy(np.concatenate([np.zeros(offset, np.uint16), a]).view(np.int16)).cuda()[offset:]
    td = torch.from_numpy(np.concatenate([np.zeros(offset, np.uint16), d]).view(np.int16)).cuda()[offset:]
    s = gpu.error_stats(ta, td)
    a64, d64 = a.astype(np.float64), d.astype(np.float64)
    err = np.abs(d64 - a64)
    assert s["n"] == n and s["max_abs_err"] == int(err.max())
    assert s["sum_sq_err"] == int((err.astype(np.int64) ** 2).sum())
    assert s["min_orig"] == int(a.min()) and s["max_orig"] == int(a.max())
    mse = (err ** 2).mean()
    rng_ = a64.max() - a64.min()
    if mse > 0 and rng_ > 0:
        assert s["psnr"] == pytest.approx(20 * np.log10(rng_) - 10 * np.log10(mse), rel=1e-12)
        assert s["nrmse"] == pytest.approx(np.sqrt(mse) / rng_, rel=1e-12)
    nz = a64 != 0
    if nz.any():
        assert s["max_rel_err"] == pytest.approx((err[nz] / a64[nz]).max(), rel=1e-6)
    # normErr = sqrt(sum err^2), normErr_norm = normErr / sqrt(sum dec^2)
    # (cuLSZ_utility.cu:900, 935-936: sum22 accumulates the decoded values)
    norm = np.sqrt((err ** 2).sum())
    assert s["norm_err"] == pytest.approx(norm, rel=1e-12)
    dsq = (d64 ** 2).sum()
    if dsq > 0:
        assert s["norm_err_norm"] == pytest.approx(norm / np.sqrt(dsq), rel=1e-12)


def test_metrics_of_a_lossy_round_trip(gpu):
    import torch
    vol = synth("cssi", (4, 256, 520), seed=3)
    d = torch.from_numpy(vol.view(np.int16)).cuda()
    out, n = gpu.compress(d, vol.shape, (1, 1, 1, 1), 1.0)
    s = gpu.error_stats(d, gpu.decompress(out, n, vol.shape))
    assert s["max_abs_err"] == 0 and s["sum_sq_err"] == 0
    out, n = gpu.compress(d, vol.shape, (3, 5, 10, 15), 1.0)        # no pooling: error < bin
    s = gpu.error_stats(d, gpu.decompress(out, n, vol.shape, (3, 5, 10, 15)))
    assert 0 < s["max_abs_err"] <= 14 and np.isfinite(s["psnr"])


@pytest.mark.gpu
@pytest.mark.parametrize("nbytes", [16, 1000, 4096 + 7, 3 * 1024 * 1024 + 5])
def test_copy_bytes(gpu, nbytes):
    """The calibration copy reproduces its source exactly, tail bytes included,
    and leaves the bytes after the destination alone."""
    import torch
    src = torch.randint(0, 256, (nbytes,), dtype=torch.uint8, device="cuda")
    dst = torch.full((nbytes + 32,), 7, dtype=torch.uint8, device="cuda")
    gpu.copy_bytes(dst[:nbytes], src)
    torch.cuda.synchronize()
    assert torch.equal(dst[:nbytes], src)
    assert bool((dst[nbytes:] == 7).all())
    with pytest.raises(ValueError):
        gpu.copy_bytes(dst[:nbytes - 1], src)
    with pytest.raises(gpu.LscompError):
        gpu.copy_bytes(dst[1:nbytes + 1], src)   # misaligned destination


# ---- SSIM (cuLSZ_utility.cu:757-886) against the oracle's restatement --------

def _noisy(a, rng, amp):
    return np.clip(a.astype(np.int64) + rng.integers(-amp, amp + 1, a.shape), 0, 65535).astype(np.uint16)


def _dev(v):
    import torch
    return torch.from_numpy(np.ascontiguousarray(v).view(np.int16)).cuda()


# one window; tiles of 61 x 8 windows along z, y and chunks of up to 32 along x,
# with odd and even remainders; a shape whose windows end one short of z
@pytest.mark.parametrize("shape", [(7, 7, 7), (9, 20, 140), (20, 33, 300), (140, 9, 9), (8, 14, 8), (11, 7, 270)],
                         ids=lambda s: "x".join(map(str, s)))
def test_ssim_vs_oracle(gpu, orc, shape):
    rng = np.random.default_rng(sum(shape))
    a = rng.integers(0, 65536, shape).astype(np.uint16)
    b = _noisy(a, rng, 2000)
    got, want = gpu.ssim(_dev(a), _dev(b), shape), orc.ssim(a, b)
    assert got == pytest.approx(want, rel=1e-10, abs=1e-13)


def test_ssim_of_lossy_round_trips(gpu, orc):
    """CSSI- and XPCS-like frames through the codec: sparse data, windows whose
    original is constant (range 0), and the decoded volume's quantization."""
    for kind, shape, bins, p in (("cssi", (12, 200, 260), (3, 5, 10, 15), 0.5),
                                 ("xpcs", (9, 64, 520), (3, 3, 3, 3), 0.5),
                                 ("cssi", (10, 90, 77), (10, 10, 10, 10), 1.0)):
        vol = synth(kind, shape, seed=9)
        d = _dev(vol)
        out, n = gpu.compress(d, shape, bins, p)
        dec = gpu.decompress(out, n, shape, bins)
        got = gpu.ssim(d, dec, shape)
        want = orc.ssim(vol, dec.cpu().numpy().view(np.uint16))
        assert got == pytest.approx(want, rel=1e-10, abs=1e-13), kind


def test_ssim_medium_volume(gpu, orc):
    """40 x 300 x 400: 492 k windows, many workgroups and chunks."""
    shape = (40, 300, 400)
    rng = np.random.default_rng(40)
    a = synth("xpcs", shape, seed=40)
    b = _noisy(a, rng, 3)
    got, want = gpu.ssim(_dev(a), _dev(b), shape), orc.ssim(a, b)
    assert got == pytest.approx(want, rel=1e-10, abs=1e-13)


def test_ssim_identity_at_full_frame_size(gpu):
    """SSIM(v, v) = 1 and a lossless round trip gives 1, on 64 CSSI frames of
    1813 x 1558 (20 M windows)."""
    shape = (64, 1813, 1558)
    vol = synth("cssi", shape, seed=2)
    d = _dev(vol)
    assert abs(gpu.ssim(d, d, shape) - 1.0) < 1e-12
    out, n = gpu.compress(d, shape, (1, 1, 1, 1), 1.0)
    assert abs(gpu.ssim(d, gpu.decompress(out, n, shape), shape) - 1.0) < 1e-12


# rows at every alignment of both volumes (odd widths alternate), the first and
# last rows read by elements, values of 14 bits with and without one of 15 in the
# original only or the decoded volume only (the wide sums; test_ssim_narrow_limit
# has the narrow ones and their limit), windows on both sides of a wave's and a
# workgroup's
@pytest.mark.parametrize("oa,od", [(0, 0), (1, 1), (0, 1), (1, 0)])
@pytest.mark.parametrize("shape", [(7, 7, 7), (8, 21, 133), (13, 24, 136), (9, 11, 265)],
                         ids=lambda s: "x".join(map(str, s)))
def test_ssim_alignment_and_value_range(gpu, orc, shape, oa, od):
    import torch
    rng = np.random.default_rng(oa + 2 * od + sum(shape))
    n = shape[0] * shape[1] * shape[2]
    for big in (0, 1, 2):
        a = rng.integers(0, 1 << 14, shape).astype(np.uint16)
        b = _noisy(a, rng, 50)
        b[b >= 1 << 14] = (1 << 14) - 1
        if big:
            (a if big == 1 else b)[tuple(rng.integers(0, k) for k in shape)] = 1 << 14
        va, vb = (torch.zeros(n + 8, dtype=torch.int16, device="cuda")[o:o + n] for o in (oa, od))
        va.copy_(_dev(a).view(-1))
        vb.copy_(_dev(b).view(-1))
        assert gpu.ssim(va, vb, shape) == pytest.approx(orc.ssim(a, b), rel=1e-10, abs=1e-13)


# the grouped pass and its element-wise ends: dword-aligned at different heads,
# volumes of different alignment, fewer elements than a group, sums of squares
# on both sides of 32 bits, zeros in the original (no relative error there)
@pytest.mark.parametrize("oa,od", [(0, 0), (1, 1), (0, 1), (3, 1)])
@pytest.mark.parametrize("n", [1, 8, 9, 17, 4097, 8 * 512 * 1024 + 13])
def test_metrics_alignment_and_value_range(gpu, n, oa, od):
    import torch
    rng = np.random.default_rng(n + oa)
    for top in (3, 1 << 14, 65536):
        a = rng.integers(0, top, n).astype(np.uint16)
        d = rng.integers(0, top, n).astype(np.uint16)
        va, vd = (torch.zeros(n + 8, dtype=torch.int16, device="cuda")[o:o + n] for o in (oa, od))
        va.copy_(torch.from_numpy(a.view(np.int16)))
        vd.copy_(torch.from_numpy(d.view(np.int16)))
        s = gpu.error_stats(va, vd)
        e = np.abs(d.astype(np.int64) - a)
        assert (s["max_abs_err"], s["min_orig"], s["max_orig"]) == (e.max(), a.min(), a.max())
        assert s["sum_sq_err"] == int((e * e).sum()) and s["sum_sq_dec"] == int((d.astype(np.int64) ** 2).sum())
        nz = a != 0
        want = (e[nz].astype(np.float32) / a[nz].astype(np.float32)).max() if nz.any() else np.float32(0)
        assert s["max_rel_err"] == float(want)


def test_ssim_rejects_volumes_without_a_window(gpu):
    import lscomp
    v = _dev(np.zeros((6, 10, 10), np.uint16))
    with pytest.raises(lscomp.LscompError):
        gpu.ssim(v, v, (6, 10, 10))


# a wave's 61 windows along size0 and the ones around them (61 fit in 127 and 128
# elements), the first elements of a window in the wave's last words; one to four
# chunks along size2; sums in 32 bits at their largest: values of one byte, of 12
# bits (the narrow sums' limit), of 14 and of 16
@pytest.mark.parametrize("shape", [(7, 9, 126), (8, 9, 127), (7, 10, 128), (9, 8, 129), (7, 9, 130), (7, 23, 251),
                                   (45, 9, 131)], ids=lambda s: "x".join(map(str, s)))
def test_ssim_wave_edges_and_products(gpu, orc, shape):
    rng = np.random.default_rng(sum(shape))
    for top in (2, 1 << 8, 1 << 12, 1 << 14, 1 << 16):
        a = rng.integers(0, top, shape).astype(np.uint16)
        b = rng.integers(0, top, shape).astype(np.uint16)
        for x, y in ((a, b), (np.full_like(a, top - 1), b), (a, a)):
            got, want = gpu.ssim(_dev(x), _dev(y), shape), orc.ssim(x, y)
            assert got == pytest.approx(want, rel=1e-10, abs=1e-13), top


# rows of more than 2^31 elements: 210 GB, the decoded volume the original's own
# memory some elements on, zeros but for values in the last columns.  A window of
# zeros has an SSIM of 1 exactly, so the sum over all windows is their number and
# what the last columns' windows lack; sums of 2^30 terms of at most 1 in doubles
# are good to 2^30 * 2^-53 * some tens, below 1e-5.
@pytest.mark.parametrize("shift", [2, 1], ids=["even", "odd"])
def test_ssim_rows_beyond_2_31(gpu, orc, shift):
    import torch
    z, w = (1 << 31) + 100, 164
    n = 49 * z
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 2 * n + (2 << 30):
        pytest.skip("needs 210 GB of free device memory")
    rng = np.random.default_rng(shift)
    small = np.zeros((7, 7, w), np.uint16)
    small[:, :, w - 90:] = rng.integers(0, 4000, (7, 7, 90))
    dec = np.zeros_like(small)
    dec[:, :, :w - shift] = small[:, :, shift:]
    buf = torch.zeros(n + 8, dtype=torch.int16, device="cuda")
    buf[:n].view(7, 7, z)[:, :, z - w:].copy_(torch.from_numpy(small.view(np.int16)))
    windows, last = (z - 7) // 2 + 1, (w - 7) // 2 + 1
    got = gpu.ssim(buf[:n], buf[shift:n + shift], (7, 7, z))
    del buf
    torch.cuda.empty_cache()
    lack = last * (1.0 - orc.ssim(small, dec))
    assert lack > 1.0
    assert windows * (1.0 - got) == pytest.approx(lack, abs=1e-4)


# the narrow sums (every value of a wave's plane below 2^12) at every alignment of
# both volumes, and their limit: one value of 4095 or 4096 in the original or the
# decoded volume only, in a corner, inside, or in a plane between, so that narrow
# and wide planes meet in a window
@pytest.mark.parametrize("oa,od", [(0, 0), (1, 1), (0, 1), (1, 0)])
@pytest.mark.parametrize("shape", [(7, 7, 7), (8, 21, 133), (13, 24, 136), (9, 11, 265)],
                         ids=lambda s: "x".join(map(str, s)))
def test_ssim_narrow_limit(gpu, orc, shape, oa, od):
    import torch
    rng = np.random.default_rng(oa + 2 * od + sum(shape))
    n = shape[0] * shape[1] * shape[2]
    va, vb = (torch.zeros(n + 8, dtype=torch.int16, device="cuda")[o:o + n] for o in (oa, od))
    places = [(0, 0, 0), tuple(k - 1 for k in shape), tuple(k // 2 for k in shape), (shape[0] // 2, 0, shape[2] - 1)]
    for at in places:
        for who, top in ((None, 0), (0, 4095), (0, 4096), (1, 4095), (1, 4096)):
            a = rng.integers(0, 4000, shape).astype(np.uint16)
            b = np.minimum(_noisy(a, rng, 50), 4094).astype(np.uint16)
            if who is not None:
                (a, b)[who][at] = top
            va.copy_(_dev(a).view(-1))
            vb.copy_(_dev(b).view(-1))
            assert gpu.ssim(va, vb, shape) == pytest.approx(orc.ssim(a, b), rel=1e-10, abs=1e-13), (at, who, top)
